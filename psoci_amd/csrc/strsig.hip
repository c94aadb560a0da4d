// String-driven direct sigma on the GPU (the plan and its index arithmetic
// are in ras.hpp / ras.cpp).
//
// Replaces, for RAS spaces (full CI and MR-CISD lists) and parts of them, the direct
// path of the reference (matrixVectorProductsScatterAccumulateLowLevel...
// DirectFetch, PsociGAhamiltonian.C:7549-7823, with matrixVectorUpdate
// :13036-13115), which regenerates every configuration-pair block.  One
// sigma call of K columns is, per chunk of KC <= 16 columns (FP64: 8 when
// device memory is short):
//   k_ras_x2c   SEF vectors -> determinant vectors, both signs (each
//               determinant belongs to one SEF: a scatter without collisions;
//               a product reads an entry of either sign without arithmetic);
//   k_ras_gemm  per tile of the compact products (RasCmp, ras.hpp): W[row]
//               [p-pair][KC] = sum over q-pairs of G[p-pair][q-pair]
//               D[row][q-pair][KC], D gathered from c into LDS through the
//               signed row of each entry (built once from the string addition
//               tables by k_ras_didx), the product on MFMA
//               (v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64);
//   k_ras_y     per SEF and column: y = scale * sum of +-W over the RI
//               terms of its determinants (the term list -- signed W offsets
//               -- is built once at setup by k_ras_terms), written once (a
//               gather: deterministic, no atomics).
// HBM layout: c [2 ndet + 1][KC] (64 B per row at KC = 16 FP32; every +c, then
// every -c, then a zero row) and W [group][pair][row][KC], so that the
// determinants that consecutive rows of a product gather, and the W terms of
// consecutive SEFs (in the order of k_ras_order), share cache lines: on 10 +
// 24 orbitals, 8 electrons, 16 FP32 columns, L2 misses of the products 95 ->
// 77 GB and of k_ras_y 43 -> 35 GB against +c and -c side by side, W
// [row][pair] and the list's own order.
#include <algorithm>
#include <cstdlib>

#include "ctx.hpp"
#include "ras.hpp"

namespace psoci {

namespace {

constexpr int kMT = 128;  // (row, column) values per product tile
constexpr int kQC = 16;   // q-pairs per LDS chunk

inline unsigned nblk(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 op(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // row of the 16x16 output held by accumulator t of lane l
  static __device__ __forceinline__ int row(int t, int l) { return 4 * (l >> 4) + t; }
};
template <>
struct Mfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 op(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int t, int l) { return 4 * t + (l >> 4); }
};

// determinant d of a SEF, or -1 outside the plan (never, for a plan that
// passes its host checks)
__device__ __forceinline__ int64_t ras_sef_det(const RasView& v, const RasSef& e, int d) {
  const RasSectorDev& S = v.sec[e.sec[d]];
  const int ca = ras_cls_of(v, S.na, e.a[d]), cb = ras_cls_of(v, S.nb, e.b[d]);
  const int64_t det =
      ras_det(v, e.sec[d], ca, e.a[d] - v.lev[S.na].cls_off[ca], cb, e.b[d] - v.lev[S.nb].cls_off[cb]);
  return det >= 0 && det < v.ndet ? det : -1;
}

// The order in which the scatter and the gather walk the SEFs (built once):
// by the lower of their determinants.  Consecutive SEFs then differ in the
// external part of one string, as do consecutive rows of a product's group,
// so a wavefront's determinant rows and W terms are consecutive in memory (a
// list in file order puts such SEFs far apart).  k_ras_mark: flag and SEF of
// each such determinant; k_ras_order: order[rank] = SEF.
__global__ __launch_bounds__(256) void k_ras_mark(const RasView* __restrict__ vp, int64_t* __restrict__ flag,
                                                  int32_t* __restrict__ sef) {
  const RasView& v = *vp;
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= v.nsef) return;
  const RasSef e = v.sef[s];
  int64_t k = ras_sef_det(v, e, 0);
  if (e.n > 1) {
    const int64_t k1 = ras_sef_det(v, e, 1);
    k = k1 < k ? k1 : k;
  }
  if (k < 0) return;
  flag[k] = 1;
  sef[k] = (int32_t)s;
}
__global__ __launch_bounds__(256) void k_ras_order(int64_t ndet, const int64_t* __restrict__ flag,
                                                   const int64_t* __restrict__ rank, const int32_t* __restrict__ sef,
                                                   int32_t* __restrict__ order) {
  const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d < ndet && flag[d]) order[rank[d]] = sef[d];
}
// The signed rows of every SEF's determinant coefficients, in that order
// (built once): rows.x = det + negative * ndet of its first determinant; rows.y
// the same for the second, or -1 (one determinant, coefficient 1/sqrt(2)) or -2
// (a closed shell, coefficient 1); -3 marks a determinant outside the plan.
__global__ __launch_bounds__(256) void k_ras_sefrows(const RasView* __restrict__ vp,
                                                     const int32_t* __restrict__ order, int2* __restrict__ rows) {
  const RasView& v = *vp;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= v.nsef) return;
  const RasSef e = v.sef[order[i]];
  int r[2] = {-3, (e.flag[0] & 2) ? -2 : -1};
  for (int d = 0; d < e.n; ++d) {
    const int64_t det = ras_sef_det(v, e, d);
    r[d] = det >= 0 ? (int)(det + (e.flag[d] & 1) * v.ndet) : -3;
  }
  rows[i] = make_int2(r[0], r[1]);
}

// c[row][KC] = +-magnitude * x[sef][col0 + q] (zero for q >= kw) for both
// signed rows (det, and ndet + det: -c_det) of each of the SEF's
// determinants; the zero row 2 ndet.  Threads follow the SEF order of k_ras_y,
// whose determinants are consecutive, so the four row writes per SEF stream
// and only the one read is scattered.  X may be wider than T (FP64 vectors
// rounded to the FP32 computation on the fly).
template <typename T, int KC, typename TX = T>
__global__ __launch_bounds__(256) void k_ras_x2c(int64_t nsef, int64_t ndet, const int32_t* __restrict__ order,
                                                 const int2* __restrict__ rows, const TX* __restrict__ X, int ldx,
                                                 int col0, int kw, T* __restrict__ c) {
  // (parts per XCD as in k_ras_y, for rows shorter than a cache line)
  const int64_t per = gridDim.x >> 3;
  const int64_t t =
      (sizeof(T) == 4 ? (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3) : (int64_t)blockIdx.x) * blockDim.x +
      threadIdx.x;
  if (t < KC) c[2 * ndet * KC + t] = (T)0;
  const int64_t i = t / KC;
  const int q = (int)(t % KC);
  if (i >= nsef) return;
  const int64_t s = order[i];
  const int2 r = rows[i];
  const T x = q < kw ? (T)X[s * (int64_t)ldx + col0 + q] : (T)0;
  const T y = (r.y == -2 ? (T)1 : (T)0x1.6a09e667f3bcdp-1) * x;
  if (r.x >= 0) {
    c[(int64_t)r.x * KC + q] = y;
    c[(r.x < ndet ? r.x + ndet : r.x - ndet) * KC + q] = -y;
  }
  if (r.y >= 0) {
    c[(int64_t)r.y * KC + q] = y;
    c[(r.y < ndet ? r.y + ndet : r.y - ndet) * KC + q] = -y;
  }
}

// Determinants of a list that is only part of its space: flags of those that
// belong to a SEF, the others' list, and their zeros (both signed rows)
__global__ __launch_bounds__(256) void k_ras_present(const RasView* __restrict__ vp, int64_t* __restrict__ absent) {
  const RasView& v = *vp;
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= v.nsef) return;
  const RasSef e = v.sef[s];
  for (int d = 0; d < e.n; ++d) {
    const int64_t k = ras_sef_det(v, e, d);
    if (k >= 0) absent[k] = 0;
  }
}
__global__ __launch_bounds__(256) void k_ras_fill64(int64_t n, int64_t* __restrict__ p, int64_t x) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = x;
}
__global__ __launch_bounds__(256) void k_ras_absent(int64_t ndet, const int64_t* __restrict__ absent,
                                                    const int64_t* __restrict__ rank, int32_t* __restrict__ list) {
  const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d < ndet && absent[d]) list[rank[d]] = (int32_t)d;
}
template <typename T, int KC>
__global__ __launch_bounds__(256) void k_ras_blank(int64_t n, int64_t ndet, const int32_t* __restrict__ list,
                                                   T* __restrict__ c) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * KC) return;
  const int64_t d = list[t / KC];
  c[d * KC + t % KC] = (T)0;
  c[(d + ndet) * KC + t % KC] = (T)0;
}

// Pair table of the compact products (built once): per block and variant the
// nqp pairs as p | r << 8 and their positions in the full product's list, -1
// for padding.
__global__ __launch_bounds__(64) void k_ras_pairs(const RasView* __restrict__ vp, int bi, int16_t* __restrict__ pr,
                                                  int16_t* __restrict__ pos) {
  const RasView& v = *vp;
  const RasCmp& C = v.cmp[bi];
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= C.nvar) return;
  int64_t oi = C.level == 0 ? 0 : g, ii = 0;
  if (C.level == 2) {
    if (C.tri) {
      ras_tri_uw(g, C.nIo, oi, ii);
    } else {
      oi = g / C.nIi;
      ii = g % C.nIi;
    }
  }
  uint64_t op, ir;
  ras_cmp_drop(v, C, oi, ii, op, ir);
  const int16_t* __restrict__ px = v.pidx + (int64_t)((C.kind ? 1 : 0) * (v.m + 1) + C.budget) * v.nbf * v.nbf;
  ras_cmp_pairs(v, C, op, ir, [&](int j, int p, int r) {
    if (j >= C.nq) return;
    pr[g * C.nqp + j] = (int16_t)(p | (r << 8));
    pos[g * C.nqp + j] = px[p * v.nbf + r];
  });
  for (int j = C.nq; j < C.nqp; ++j) pr[g * C.nqp + j] = pos[g * C.nqp + j] = -1;
}

// The variants' integral matrices, gathered from the block's full matrix
// (np x np); zero rows and columns for padding.  (A grid of at most kGvarGrid
// workgroups: a block's variants can hold more than the 2^32 elements that one
// launch may have threads, 52 GB of matrices.)
constexpr unsigned kGvarGrid = 1u << 20;
__global__ __launch_bounds__(256) void k_ras_gvar(int64_t gbase, int64_t n, int nqp, int np,
                                                  const int16_t* __restrict__ pos, const double* __restrict__ full,
                                                  double* __restrict__ g64, float* __restrict__ g32) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = e / nqp;  // variant * nqp + p-pair
    const int i = pos[row], j = pos[row / nqp * nqp + e % nqp];
    const double x = (i < 0 || j < 0) ? 0.0 : full[(int64_t)i * np + j];
    g64[gbase + e] = x;
    g32[gbase + e] = (float)x;
  }
}

// Signed vector row of every D entry (built once): didx[dbase + row * nqp +
// j] = det + negative * ndet for live pair j of row `row`, the zero row 2
// ndet when the pair cannot be added to the row's strings (ras_d_det).
__global__ __launch_bounds__(256) void k_ras_didx(const RasView* __restrict__ vp, int bi,
                                                  const int16_t* __restrict__ pr, int32_t* __restrict__ didx) {
  const RasView& v = *vp;
  const RasBlockDev& B = v.blk[bi];
  const RasCmp& C = v.cmp[bi];
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= C.nrows * C.nqp) return;
  const int64_t row = e / C.nqp;
  const int j = (int)(e % C.nqp);
  int64_t o, i;
  ras_cmp_unrow(C, row, o, i);
  const int16_t qs = pr[ras_cmp_var(C, o / C.nEo, i / C.nEi) * C.nqp + j];
  const int64_t u = C.swap ? C.i0 + i : C.o0 + o, w = C.swap ? C.o0 + o : C.i0 + i;
  int neg = 0;
  const int64_t det = qs < 0 ? -1 : ras_d_det(v, C.kind, C.sector, B.lu, B.lw, u, w, qs & 0xff, (qs >> 8) & 0xff, neg);
  didx[C.dbase + e] = (det < 0 || det >= v.ndet) ? (int32_t)(2 * v.ndet) : (int32_t)(det + neg * v.ndet);
}

// A W element: FP64 past the caches (W is read once, by k_ras_y, long after;
// 10 + 24 orbitals, 16 columns: products 42.5 -> 42.3, gather 9.4 -> 8.2 ms);
// FP32 through them (its half-line stores merge in L2: 22.9 against 23.3 ms)
__device__ __forceinline__ void ras_store(double x, double* p) { __builtin_nontemporal_store(x, p); }
__device__ __forceinline__ void ras_store(float x, float* p) { *p = x; }

// One group of rows with its matrix, and its first tile per chunk width
// (built on the host; the tile table is written from it).
struct RasGroup {
  int64_t g, w, d, rows;
  int32_t nqp, nq, pt, pad;
  int64_t tile0[4];
};

// Tiles of every group for one chunk width (rt rows per tile): row tiles
// major, the p-tiles that gather the same c rows next to each other.
__global__ __launch_bounds__(64) void k_ras_tiles(const RasGroup* __restrict__ grp, int which, int rt,
                                                  RasTile* __restrict__ out) {
  const RasGroup G = grp[blockIdx.x];
  // the p-subtiles of 16 spread evenly over the p-tiles
  const int ns = G.nqp / 16, npt = (G.nqp + G.pt - 1) / G.pt, each = ns / npt, more = ns % npt;
  const int64_t n = (G.rows + rt - 1) / rt * npt;
  for (int64_t t = threadIdx.x; t < n; t += blockDim.x) {
    const int64_t r0 = t / npt * rt;
    // (the p-tiles of a row tile differ by a subtile: their order, and the
    // wavefront pair that takes the larger half, rotate from row tile to row
    // tile so that no shader engine or SIMD always gets the longer ones)
    const int64_t turn = blockIdx.x + t / npt;
    const int pt = (int)((t + turn) % npt);
    RasTile T;
    T.g = G.g;
    T.w = G.w + r0;
    T.rows = (int32_t)G.rows;
    T.flip = (int32_t)((turn / npt) & 1);
    T.d = G.d + r0 * G.nqp;
    T.nqp = G.nqp;
    T.p0 = (uint16_t)(16 * (pt * each + (pt < more ? pt : more)));
    T.nrows = (uint8_t)(G.rows - r0 < rt ? G.rows - r0 : rt);
    T.niv = (uint8_t)(G.pt <= 64 ? G.nq : each + (pt < more ? 1 : 0));
    out[G.tile0[which] + t] = T;
  }
}

// wavefronts per SIMD the product is compiled for (a register budget: the
// compiler would otherwise hold more k-steps' operands in flight than
// occupancy can afford)
template <typename T>
constexpr int ras_lds_waves() {
  return sizeof(T) == 8 ? 3 : 6;
}

template <int N>
struct IntC {
  static constexpr int value = N;
};

// 16 bytes from this lane's global address to LDS at byte address lds + 16
// * lane (lds uniform over the wavefront); completion is counted by vmcnt.  Written as
// asm statements so that the compiler, which cannot tell the two LDS
// stages apart, does not wait for every copy in flight before each LDS read:
// the kernel waits for its copies itself (vmcnt(0) before the barrier that
// publishes a stage).  M0 carries the LDS address; nothing else in the
// kernels that use this keeps a value in M0.  A copy may not issue in the
// instruction after the one that writes M0 (one wait state: the s_nop, which
// the compiler does not add inside asm).
__device__ __forceinline__ void lds_copy16(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
}
// the same from a uniform base plus this lane's byte offset
__device__ __forceinline__ void lds_copy16(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds)
               : "memory", "m0");
}
// LDS byte address of a __shared__ location, uniform over the wavefront
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p);
}

// The products of PT <= 64 p-pairs (nqp = PT): one workgroup per tile (PT
// p-pairs x 128 (row, column) values; RasTile), four wavefronts of PT x 32
// values (PT / 16 x 2 MFMA tiles).  Operands are copied straight from global memory into LDS
// (global_load_lds_dwordx4: each lane names its own 16-byte source, the
// wavefront's 64 pieces land contiguously at one LDS address), into two LDS
// stages: the copies of chunk n + 1 are in flight while the MFMA steps
// consume chunk n, with one barrier per chunk and no staging registers.
// Layouts in LDS:
//   G stage [q][PT] -- q-pair rows of the tile's p-pairs, read from G's q
//     rows (G is symmetric, so row q holds column q); at FP32 the 16-byte
//     pieces of odd rows swap halves of every 128 bytes when PT / 16 is even,
//     which keeps the two rows one 32-lane operand read touches in separate
//     banks;
//   D stage [wavefront][q][32] -- the wavefront's rows x KC columns for each
//     q (the halves of 16 swapped for odd q, for the same reason), each
//     (row, q) entry copied from its signed row of c (the zero row for a
//     missing determinant), so no arithmetic touches the operands between
//     the copy and the MFMA; one layout for every KC whose row of c is a
//     whole number of 16-byte pieces (narrower blocks run at 4 FP32 or 2
//     FP64 columns).
// A tile's rows past its group's last repeat that row (not stored).  The
// chunk loop is unrolled over the two stages, so every LDS address is a
// constant offset, and the matrix and index addresses advance in scalar
// registers.
// One launch covers every block of one tile width (27 blocks on 10 + 24
// orbitals, 8 electrons: 5 launches instead of 27), heavy tiles first; tiles
// are dealt to the 8 XCDs in runs of 2^sh, so that the tiles of a row group
// (the same c rows and matrix) share an L2.
template <typename T, int KC, int PT, int WPE = ras_lds_waves<T>()>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE)))
void k_ras_gemm(const RasTile* __restrict__ tiles, int64_t ntiles, int sh, const int32_t* __restrict__ didx,
                const T* __restrict__ G, const T* __restrict__ c, T* __restrict__ W) {
  typedef Mfma<T> M;
  typedef typename M::v4 v4;
  constexpr int RT = kMT / KC;           // rows per tile
  constexpr int RW = RT / 4;             // rows per wavefront
  constexpr int NI = PT / 16;            // p-subtiles per wavefront
  constexpr int SL = 16 / sizeof(T);     // values per 16-byte piece
  constexpr int SPE = KC / SL;           // pieces per D entry
  constexpr int DI = 32 * kQC / (64 * SL);  // D copies per wavefront and chunk
  constexpr int GSR = PT / SL;           // pieces per G row
  constexpr int GI = kQC * GSR / 64;     // G copies per chunk
  constexpr int GW = (GI + 3) / 4;       // G copies per wavefront (at most)
  constexpr bool SWZ = sizeof(T) == 4 && (PT / 16) % 2 == 0;
  static_assert(KC % SL == 0 && RW >= 2 && kQC * GSR % 64 == 0, "copy shapes");
  __shared__ __align__(16) T Gs[2][kQC * PT];
  __shared__ __align__(16) T Ds[2][kQC * kMT];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t b = blockIdx.x >> 3;
  const int64_t ti = ((((b >> sh) << 3) + (blockIdx.x & 7)) << sh) + (b & ((1 << sh) - 1));
  if (ti >= ntiles) return;  // uniform per workgroup
  const RasTile tile = tiles[ti];
  const int nrows = tile.nrows, nq = tile.niv;
  constexpr int nch = PT / kQC;

  // this lane's sources: its D entries' offsets in the index table and its G
  // pieces' byte offsets, both from bases that advance by a chunk
  const int32_t* __restrict__ dx = didx + tile.d;
  const T* __restrict__ Gb = G + tile.g;
  uint32_t dxo[DI];
#pragma unroll
  for (int d = 0; d < DI; ++d) {
    const int slot = d * 64 + lane;
    const int q = slot / (SPE * RW), r = ((slot / SPE) % RW) ^ ((q & 1) * (RW / 2));
    const int row = RW * wave + r;
    dxo[d] = (uint32_t)((row < nrows ? row : nrows - 1) * PT + q);
  }
  uint32_t go[GW];
#pragma unroll
  for (int gi = 0; gi < GW; ++gi) {
    const int sl = 64 * (wave + 4 * gi) + lane, k = sl / GSR;
    const int r = SWZ ? (sl % GSR) ^ (4 * (k & 1)) : sl % GSR;
    go[gi] = (uint32_t)((k * PT + r * SL) * sizeof(T));
  }
  const T* __restrict__ cl = c + SL * (lane % SPE);
  // LDS addresses of this wavefront's first D copy and first G copy (stage 0)
  const uint32_t dl0 = lds_addr(&Ds[0][32 * kQC * wave]);
  const uint32_t gl0 = lds_addr(&Gs[0][64 * wave * SL]);
  auto fetch_idx = [&](int32_t (&ix)[DI]) {
#pragma unroll
    for (int d = 0; d < DI; ++d) ix[d] = dx[dxo[d]];
    dx += kQC;
  };
  // the copies of the next chunk into stage ST: D pieces first (they use the
  // indices loaded a chunk earlier), then G
  auto issue = [&](auto stc, const int32_t (&ix)[DI]) {
    constexpr int ST = decltype(stc)::value;
    // every source address is formed (its index load waited for) before
    // the first copy issues: a wait for an index load placed between two
    // copies would also wait for the copy before it
    const T* src[DI];
#pragma unroll
    for (int d = 0; d < DI; ++d) src[d] = cl + (uint64_t)(uint32_t)ix[d] * KC;
#pragma unroll
    for (int d = 0; d < DI; ++d) asm volatile("" : "+v"(src[d]));
#pragma unroll
    for (int d = 0; d < DI; ++d)
      lds_copy16(src[d], dl0 + (uint32_t)((ST * kQC * kMT + d * 64 * SL) * sizeof(T)));
#pragma unroll
    for (int gi = 0; gi < GW; ++gi) {
      if (wave + 4 * gi >= GI) continue;
      lds_copy16(Gb, go[gi], gl0 + (uint32_t)((ST * kQC * PT + 64 * 4 * gi * SL) * sizeof(T)));
    }
    Gb += kQC * PT;
  };

  // lane offsets of the MFMA operand reads (k row kr = lane / 16 within a
  // step): p-subtile i of G sits at a0[i & 1] + 16 i (with the swap of
  // 64-byte halves on odd rows: 16 (i ^ 1) = 16 i -+ 16); value subtile j of
  // D at b0[j] (its halves swapped on odd rows)
  const int kr = lane >> 4, l15 = lane & 15;
  const int sw = SWZ ? 16 * (kr & 1) : 0;
  const int a0[2] = {kr * PT + l15 + sw, kr * PT + l15 - sw};
  const int b0[2] = {32 * (kQC * wave + kr) + l15 + 16 * (kr & 1), 32 * (kQC * wave + kr) + l15 + 16 - 16 * (kr & 1)};

  v4 acc[NI][2];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = v4{0, 0, 0, 0};
  int32_t ixn[DI];
  fetch_idx(ixn);
  issue(IntC<0>{}, ixn);
  if (nch > 1) fetch_idx(ixn);
  // one chunk on stage ST; `left` chunks follow
  auto chunk = [&](auto stc, int left) {
    constexpr int ST = decltype(stc)::value;
    // this wavefront's copies of the chunk have landed, every wavefront's
    // have after the barrier, and the other stage is free (its reads ended
    // before the barrier)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (left > 0) {
      issue(IntC<1 - ST>{}, ixn);
      if (left > 1) fetch_idx(ixn);
    }
    const T* __restrict__ gs = Gs[ST];
    const T* __restrict__ ds = Ds[ST];
#pragma unroll
    for (int kk = 0; kk < kQC / 4; ++kk) {
      T a[NI], bb[2];
#pragma unroll
      for (int i = 0; i < NI; ++i) a[i] = gs[a0[i & 1] + 16 * i + 4 * kk * PT];
#pragma unroll
      for (int j = 0; j < 2; ++j) bb[j] = ds[b0[j] + 4 * kk * 32];
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = M::op(a[i], bb[j], acc[i][j]);
    }
  };
  for (int left = nch - 1; left >= 0; left -= 2) {
    chunk(IntC<0>{}, left);
    if (left > 0) chunk(IntC<1>{}, left - 1);
  }
  T* __restrict__ Wt = W + tile.w * KC;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int m = 16 * j + l15, row = RW * wave + m / KC;
    if (row >= nrows) continue;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int p = 16 * i + M::row(t, lane);
        if (p < nq) ras_store(acc[i][j][t], &Wt[((int64_t)p * tile.rows + row) * KC + m % KC]);
      }
  }
}

// The products of more than 64 p-pairs: one workgroup per tile of up to 128
// p-pairs x 128 (row, column) values, four wavefronts as 2 x 2 of up to 64 x 64
// (the first pair of wavefronts takes the first half of the tile's n
// p-subtiles of 16, the other pair the rest).  Against k_ras_gemm's 64 x 128
// tiles a D piece is gathered by half as many tiles and an LDS operand feeds
// four MFMAs instead of 2.7.  Copies, stages and chunk loop as in k_ras_gemm.
// Layouts in LDS: both stages [q][128], the 16-value groups of row q at group
// position ^ (q & 3) within their four, so that the four rows one operand
// read touches lie in separate banks; p-subtile i of the second wavefront
// pair sits at group 4 + i.
template <typename T, int KC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : 3)))
void k_ras_gemm_wide(const RasTile* __restrict__ tiles, int64_t ntiles, int sh, const int32_t* __restrict__ didx,
                     const T* __restrict__ G, const T* __restrict__ c, T* __restrict__ W) {
  typedef Mfma<T> M;
  typedef typename M::v4 v4;
  constexpr int SL = 16 / sizeof(T);       // values per 16-byte piece
  constexpr int PR = kMT / SL;             // pieces per LDS row
  constexpr int NC = kQC * PR / 256;       // copies of each operand per wavefront and chunk
  static_assert(KC % SL == 0, "copy shapes");
  __shared__ __align__(16) T Gs[2][kQC * kMT];
  __shared__ __align__(16) T Ds[2][kQC * kMT];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t b = blockIdx.x >> 3;
  const int64_t ti = ((((b >> sh) << 3) + (blockIdx.x & 7)) << sh) + (b & ((1 << sh) - 1));
  if (ti >= ntiles) return;  // uniform per workgroup
  const RasTile tile = tiles[ti];
  const int nrows = tile.nrows, nqp = tile.nqp, p0 = tile.p0;
  const int n0 = (tile.niv + 1) >> 1, n1 = tile.niv >> 1;  // p-subtiles of the two wavefront pairs
  const int nch = nqp / kQC;

  // this lane's sources (as in k_ras_gemm): copy d of the wavefront fills the
  // pieces 64 (wave + 4 d) + lane of a stage
  const int32_t* __restrict__ dx = didx + tile.d;
  const T* __restrict__ Gb = G + tile.g + p0;
  uint32_t dxo[NC], go[NC];
  int vo = 0;  // column of the lane's pieces (the same for every copy)
#pragma unroll
  for (int d = 0; d < NC; ++d) {
    const int sl = 64 * (wave + 4 * d) + lane, q = sl / PR;
    const int v = ((sl % PR) * SL) ^ (16 * (q & 3));
    const int row = v / KC;
    dxo[d] = (uint32_t)((row < nrows ? row : nrows - 1) * nqp + q);
    vo = v % KC;
    const int sp = v >> 4, sub = sp < 4 ? (sp < n0 ? sp : 0) : (sp - 4 < n1 ? n0 + sp - 4 : 0);
    go[d] = (uint32_t)((q * nqp + 16 * sub + (v & 15)) * sizeof(T));
  }
  const T* __restrict__ cl = c + vo;
  const uint32_t dl0 = lds_addr(&Ds[0][64 * wave * SL]);
  const uint32_t gl0 = lds_addr(&Gs[0][64 * wave * SL]);
  auto fetch_idx = [&](int32_t (&ix)[NC]) {
#pragma unroll
    for (int d = 0; d < NC; ++d) ix[d] = dx[dxo[d]];
    dx += kQC;
  };
  auto issue = [&](auto stc, const int32_t (&ix)[NC]) {
    constexpr int ST = decltype(stc)::value;
    const T* src[NC];
#pragma unroll
    for (int d = 0; d < NC; ++d) src[d] = cl + (uint64_t)(uint32_t)ix[d] * KC;
#pragma unroll
    for (int d = 0; d < NC; ++d) asm volatile("" : "+v"(src[d]));
#pragma unroll
    for (int d = 0; d < NC; ++d)
      lds_copy16(src[d], dl0 + (uint32_t)((ST * kQC * kMT + d * 256 * SL) * sizeof(T)));
#pragma unroll
    for (int d = 0; d < NC; ++d)
      lds_copy16(Gb, go[d], gl0 + (uint32_t)((ST * kQC * kMT + d * 256 * SL) * sizeof(T)));
    Gb += (int64_t)kQC * nqp;
  };
  const int kr = lane >> 4, l15 = lane & 15, wr = (wave >> 1) ^ tile.flip, wc = wave & 1;
  int a0[4], b0[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a0[i] = kr * kMT + 64 * wr + 16 * (i ^ kr) + l15;
    b0[i] = kr * kMT + 64 * wc + 16 * (i ^ kr) + l15;
  }

  auto run = [&](auto nvc) {
    constexpr int NV = decltype(nvc)::value;
    v4 acc[NV][4];
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = v4{0, 0, 0, 0};
    int32_t ixn[NC];
    // operands of two k-steps: one is read from LDS while the other multiplies
    T a[2][NV], bb[2][4];
    auto read = [&](auto stc, auto kkc, auto setc) {
      constexpr int ST = decltype(stc)::value, kk = decltype(kkc)::value, S = decltype(setc)::value;
#pragma unroll
      for (int i = 0; i < NV; ++i) a[S][i] = Gs[ST][a0[i] + 4 * kk * kMT];
#pragma unroll
      for (int j = 0; j < 4; ++j) bb[S][j] = Ds[ST][b0[j] + 4 * kk * kMT];
    };
    auto mul = [&](auto setc) {
      constexpr int S = decltype(setc)::value;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = M::op(a[S][i], bb[S][j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    };
    // every wavefront's copies into the next stage have landed and its reads
    // of the other have ended (the copies of the chunk after go there)
    auto turn = [&](auto stc, int left) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __syncthreads();
      if (left > 0) {
        issue(stc, ixn);
        if (left > 1) fetch_idx(ixn);
      }
    };
    fetch_idx(ixn);
    issue(IntC<0>{}, ixn);
    if (nch > 1) fetch_idx(ixn);
    turn(IntC<1>{}, nch - 1);
    read(IntC<0>{}, IntC<0>{}, IntC<0>{});
    // one chunk on stage ST; `left` chunks follow.  The barrier sits before
    // the last k-step, whose operands are in registers, so that its MFMAs
    // cover the first reads of the next stage
    auto chunk = [&](auto stc, int left) {
      constexpr int ST = decltype(stc)::value;
      read(IntC<ST>{}, IntC<1>{}, IntC<1>{});
      mul(IntC<0>{});
      read(IntC<ST>{}, IntC<2>{}, IntC<0>{});
      mul(IntC<1>{});
      read(IntC<ST>{}, IntC<3>{}, IntC<1>{});
      mul(IntC<0>{});
      if (left > 0) {
        turn(IntC<ST>{}, left - 1);
        read(IntC<1 - ST>{}, IntC<0>{}, IntC<0>{});
      }
      mul(IntC<1>{});
    };
    for (int left = nch - 1; left >= 0; left -= 2) {
      chunk(IntC<0>{}, left);
      if (left > 0) chunk(IntC<1>{}, left - 1);
    }
    T* __restrict__ Wt = W + tile.w * KC;
    const int ps = p0 + (wr ? 16 * n0 : 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = 64 * wc + 16 * j + l15, row = m / KC;
      if (row >= nrows) continue;
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          ras_store(acc[i][j][t], &Wt[((int64_t)(ps + 16 * i + M::row(t, lane)) * tile.rows + row) * KC + m % KC]);
    }
  };
  // the same number of barriers in every variant: nch
  const int nv = wr ? n1 : n0;
  if (nv == 4) run(IntC<4>{});
  else if (nv == 3) run(IntC<3>{});
  else run(IntC<2>{});
}

// The term list of every SEF (built once), in the SEF order: FILL = false
// counts the terms of SEF order[s] into cnt[s]; FILL = true writes them, as the W offset per column
// with bit 31 set for a negative sign (the determinants' coefficient signs
// folded in), at toff[s] (the scanned counts), and the SEF's scale code.
template <bool FILL>
__global__ __launch_bounds__(256) void k_ras_terms(const RasView* __restrict__ vp,
                                                   const int32_t* __restrict__ order, int64_t* __restrict__ cnt,
                                                   const int64_t* __restrict__ toff, int32_t* __restrict__ term,
                                                   int8_t* __restrict__ scl, int* __restrict__ bad) {
  const RasView& v = *vp;
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= v.nsef) return;
  const RasSef e = v.sef[order[s]];
  if (!FILL) {
    int64_t n = 0;
    ras_sef_terms(v, e, bad, [&](int64_t, int) { ++n; });
    cnt[s] = n;
    return;
  }
  int64_t o = toff[s];
  const int64_t end = toff[s + 1];
  const int code = ras_sef_terms(v, e, bad, [&](int64_t off, int neg) {
    if (o >= end) {
      *bad = 1;
      return;
    }
    term[o++] = (int32_t)((uint32_t)off | ((uint32_t)neg << 31));
  });
  scl[s] = (int8_t)code;
  if (o != end) *bad = 1;
}

// y[sef][col0 + q] = scale * sum of +-W[off][q] over the SEF's terms (Y may
// be wider than T: the FP32 result widened exactly)
template <typename T, int KC, typename TY = T>
__global__ __launch_bounds__(256) void k_ras_y(const int64_t* __restrict__ toff, const int32_t* __restrict__ term,
                                               const int8_t* __restrict__ scl, const int32_t* __restrict__ order,
                                               const T* __restrict__ W, int64_t nsef,
                                               TY* __restrict__ Y, int ldy, int col0, int kw) {
  // FP32 rows are half a cache line: each XCD takes a contiguous part of the
  // SEFs, so that both halves are read through one L2 (10 + 24 orbitals, 16
  // columns: 5.4 -> 5.0 ms; whole lines, FP64: 8.2 -> 8.7 ms, so not there)
  const int64_t per = gridDim.x >> 3;
  const int64_t t =
      (sizeof(T) == 4 ? (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3) : (int64_t)blockIdx.x) * blockDim.x +
      threadIdx.x;
  const int64_t s = t / KC;
  const int q = (int)(t % KC);
  if (s >= nsef) return;
  const int64_t b = toff[s], e = toff[s + 1];
  T a0 = (T)0, a1 = (T)0;
  int64_t i = b;
  for (; i + 4 <= e; i += 4) {
    const int32_t t0 = term[i], t1 = term[i + 1], t2 = term[i + 2], t3 = term[i + 3];
    const T w0 = W[(int64_t)(t0 & 0x7fffffff) * KC + q];
    const T w1 = W[(int64_t)(t1 & 0x7fffffff) * KC + q];
    const T w2 = W[(int64_t)(t2 & 0x7fffffff) * KC + q];
    const T w3 = W[(int64_t)(t3 & 0x7fffffff) * KC + q];
    a0 += t0 < 0 ? -w0 : w0;
    a1 += t1 < 0 ? -w1 : w1;
    a0 += t2 < 0 ? -w2 : w2;
    a1 += t3 < 0 ? -w3 : w3;
  }
  for (; i < e; ++i) {
    const int32_t t0 = term[i];
    const T w0 = W[(int64_t)(t0 & 0x7fffffff) * KC + q];
    a0 += t0 < 0 ? -w0 : w0;
  }
  const int8_t sc = scl[s];
  const T f = sc == 2 ? (T)1 : (sc == 1 ? (T)0x1.6a09e667f3bcdp+0 : (T)0x1.6a09e667f3bcdp-1);
  if (q < kw) Y[order[s] * (int64_t)ldy + col0 + q] = (TY)(f * (a0 + a1));
}

// Flags a configuration pair one electron apart whose single-excitation sum
// vnt[0] is exactly zero in either orientation (bit 1), and one where an
// exchange integral (e o|o f) its elements could use is not (bit 0): the
// reference skips such a block (processSingleExcitation returns 0,
// PsociHamiltonian.C:190-261), which the determinant Hamiltonian does not.
//
// One thread per configuration and target orbital f.  complete: every pair
// is seen from both of its configurations, so one orientation each is enough.
// A thread per configuration with both loops was one long chain: 0.39 ms on
// full CI of 10 orbitals and 8 electrons (0.026 ms so), 0.86 ms on 8 + 24
// orbitals (0.17 ms), 4.4 ms on 10 + 24 (2.6 ms).
__global__ __launch_bounds__(256) void k_ras_zero_singles(int64_t ncfg, const uint64_t* __restrict__ dm,
                                                          const uint64_t* __restrict__ sm, uint64_t emask, int m,
                                                          int nbf, int complete, const double* __restrict__ one,
                                                          const double* __restrict__ two, int* __restrict__ flag) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t ci = t / nbf;
  const int f = (int)(t - ci * nbf);
  if (ci >= ncfg) return;
  const uint64_t dI = dm[ci], sI = sm[ci];
  const int nI = popc(sI);
  const uint64_t bf = 1ull << f;
  if (dI & bf) return;
  for (uint64_t ex = (dI | sI) & ~bf; ex; ex &= ex - 1) {
    const int e = ctz(ex);
    const uint64_t be = 1ull << e;
    uint64_t dJ = dI, sJ = sI;
    if (dJ & be) {
      dJ &= ~be;
      sJ |= be;
    } else {
      sJ &= ~be;
    }
    if (sJ & bf) {
      sJ &= ~bf;
      dJ |= bf;
    } else {
      sJ |= bf;
    }
    if (2 * popc(dJ & emask) + popc(sJ & emask) > m) continue;
    const int nJ = popc(sJ);
    PairInfo P1, P2;
    pair_setup(P1, 1, 0, dI, sI, nI, dJ, sJ, nJ, nbf, one, two);
    if (!complete) pair_setup(P2, 1, 0, dJ, sJ, nJ, dI, sI, nI, nbf, one, two);
    if (P1.kind != 0 && (complete || P2.kind != 0)) continue;
    if (!(*(volatile int*)flag & 2)) atomicOr(flag, 2);
    for (uint64_t o = (dI | sI | dJ | sJ) & ~be & ~bf; o; o &= o - 1) {
      const int c = ctz(o);
      if (g2(two, e, c, c, f) != 0.0) {
        atomicOr(flag, 1);
        return;
      }
    }
  }
}

// Optional per-launch events of a timed sigma: group 0 the SEF ->
// determinant scatter, 1..3 the products of each kind, 4 the SEF gather.
struct RasTiming {
  std::vector<hipEvent_t> ev;
  std::vector<int> group;  // group of the launch that ends at ev[i + 1]
  void mark(hipStream_t s, int g) {
    hipEvent_t e;
    PSOCI_HIP(hipEventCreate(&e));
    PSOCI_HIP(hipEventRecord(e, s));
    ev.push_back(e);
    if (g >= 0) group.push_back(g);
  }
  ~RasTiming() {
    for (hipEvent_t e : ev) (void)hipEventDestroy(e);
  }
};

// p-pairs per product tile: one exact tile up to 64, else k_ras_gemm_wide's
inline int ras_tile_width(int nqp) { return nqp <= 64 ? nqp : kMT; }

template <typename T, int KC, typename TIO = T>
void ras_chunk(Ctx& c, const TIO* X, int ldx, TIO* Y, int ldy, int col0, int kw, RasTiming* tm = nullptr) {
  const RasPlan& P = c.ras;
  T* cv = reinterpret_cast<T*>(c.d_rasc.p);
  T* W = reinterpret_cast<T*>(c.d_rasw.p);
  const T* G = sizeof(T) == 4 ? reinterpret_cast<const T*>(c.d_rasg32.p) : reinterpret_cast<const T*>(c.d_rasg64.p);
  const int64_t nsef = (int64_t)P.sef.size();
  if (tm && tm->ev.empty()) tm->mark(c.stream, -1);
  hipLaunchKernelGGL((k_ras_x2c<T, KC, TIO>), dim3(8 * nblk(nsef * KC, 8 * 256)), dim3(256), 0, c.stream, nsef, P.ndet,
                     c.d_rasorder.p, c.d_rasrows.p, X, ldx, col0, kw, cv);
  PSOCI_HIP(hipGetLastError());
  if (c.d_rasabsent.n) {
    const int64_t na = (int64_t)c.d_rasabsent.n;
    hipLaunchKernelGGL((k_ras_blank<T, KC>), dim3(nblk(na * KC, 256)), dim3(256), 0, c.stream, na, P.ndet,
                       c.d_rasabsent.p, cv);
    PSOCI_HIP(hipGetLastError());
  }
  if (tm) tm->mark(c.stream, 0);
  constexpr int ki = KC == 16 ? 0 : KC == 8 ? 1 : KC == 4 ? 2 : 3;
  const std::vector<RasLaunch>& L = c.ras_launch[ki];
  for (size_t i = 0; i < L.size();) {
    // every kind of one tile width in one launch; a timed sigma times them
    // one by one
    size_t e = i + 1;
    int64_t nt = L[i].ntiles;
    for (; !tm && e < L.size() && L[e].pt == L[i].pt; ++e) nt += L[e].ntiles;
    int sh = 5;  // runs of 32 tiles per XCD, shorter where they would leave XCDs idle
    while (sh > 0 && nt < (int64_t)8 * 8 << sh) --sh;
    const unsigned grid = (unsigned)(((nt + ((int64_t)8 << sh) - 1) >> (sh + 3)) << (sh + 3));
    const RasTile* tiles = c.d_rastile[ki].p + L[i].tile0;
    switch (L[i].pt) {
#define PSOCI_RAS_GEMM(PTV)                                                                                     \
  case PTV:                                                                                                     \
    hipLaunchKernelGGL((k_ras_gemm<T, KC, PTV>), dim3(grid), dim3(256), 0, c.stream, tiles, nt, sh, c.d_rasdidx.p, \
                       G, cv, W);                                                                               \
    break;
      PSOCI_RAS_GEMM(16)
      PSOCI_RAS_GEMM(32)
      PSOCI_RAS_GEMM(48)
      PSOCI_RAS_GEMM(64)
#undef PSOCI_RAS_GEMM
      default:
        hipLaunchKernelGGL((k_ras_gemm_wide<T, KC>), dim3(grid), dim3(256), 0, c.stream, tiles, nt, sh,
                           c.d_rasdidx.p, G, cv, W);
    }
    PSOCI_HIP(hipGetLastError());
    if (tm) tm->mark(c.stream, 1 + L[i].kind);
    i = e;
  }
  hipLaunchKernelGGL((k_ras_y<T, KC, TIO>), dim3(8 * nblk(nsef * KC, 8 * 256)), dim3(256), 0, c.stream, c.d_rastoff.p,
                     c.d_rasterm.p, c.d_rasscl.p, c.d_rasorder.p, W, nsef, Y, ldy, col0, kw);
  PSOCI_HIP(hipGetLastError());
  if (tm) tm->mark(c.stream, 4);
}

// T: the computation's type; TIO: the vectors' (FP64 vectors with an FP32
// computation: rounded on the way in, widened on the way out)
template <typename T, typename TIO = T>
void ras_any_k(Ctx& c, int k, const TIO* X, int ldx, TIO* Y, int ldy, RasTiming* tm = nullptr) {
  const int kmax = sizeof(T) == 4 ? 16 : c.ras_kc64;
  for (int c0 = 0; c0 < k; c0 += kmax) {
    const int kw = std::min(kmax, k - c0);
    if (kw > 8)
      ras_chunk<T, 16, TIO>(c, X, ldx, Y, ldy, c0, kw, tm);
    else if (kw > 4) ras_chunk<T, 8, TIO>(c, X, ldx, Y, ldy, c0, kw, tm);
    else if (kw > 2 || sizeof(T) == 4) ras_chunk<T, 4, TIO>(c, X, ldx, Y, ldy, c0, kw, tm);
    else if constexpr (sizeof(T) == 8) ras_chunk<T, 2, TIO>(c, X, ldx, Y, ldy, c0, kw, tm);
  }
}

}  // namespace

// Groups of every block, ordered by (tile width, kind, pairs descending), and
// the tile table and launches of each chunk width (16, 8, 4 and, for FP64, 2
// columns).
static void ras_tile_tables(Ctx& c) {
  const RasPlan& P = c.ras;
  std::vector<int> order;
  for (int bi = 0; bi < (int)P.cmp.size(); ++bi)
    if (P.cmp[bi].nq > 0) order.push_back(bi);
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
    const RasCmp &A = P.cmp[x], &B = P.cmp[y];
    const int pa = ras_tile_width(A.nqp), pb = ras_tile_width(B.nqp);
    if (pa != pb) return pa > pb;
    if (A.kind != B.kind) return A.kind < B.kind;
    return A.nqp > B.nqp;
  });
  std::vector<RasGroup> grp;
  int64_t nt[4] = {0, 0, 0, 0};
  for (int k = 0; k < 4; ++k) c.ras_launch[k].clear();
  for (int bi : order) {
    const RasCmp& C = P.cmp[bi];
    const int pt = ras_tile_width(C.nqp), npt = (C.nqp + pt - 1) / pt;
    for (int k = 0; k < 4; ++k)
      if (c.ras_launch[k].empty() || c.ras_launch[k].back().pt != pt || c.ras_launch[k].back().kind != C.kind)
        c.ras_launch[k].push_back(RasLaunch{pt, C.kind, nt[k], 0});
    ras_cmp_groups(C, [&](int64_t g, int64_t r0, int64_t rows) {
      RasGroup R;
      R.g = C.gbase + g * C.nqp * C.nqp;
      R.w = C.wbase + r0 * C.nqp;
      R.d = C.dbase + r0 * C.nqp;
      R.rows = rows;
      R.nqp = C.nqp;
      R.nq = C.nq;
      R.pt = pt;
      R.pad = 0;
      for (int k = 0; k < 4; ++k) {
        const int rt = kMT / (16 >> k);
        const int64_t n = (rows + rt - 1) / rt * npt;
        R.tile0[k] = nt[k];
        nt[k] += n;
        c.ras_launch[k].back().ntiles += n;
      }
      grp.push_back(R);
    });
  }
  DevBuf<RasGroup> dg;
  dg.upload(grp, c.stream);
  for (int k = 0; k < 4; ++k) {
    c.d_rastile[k].alloc(nt[k]);
    if (grp.empty()) continue;
    hipLaunchKernelGGL(k_ras_tiles, dim3((unsigned)grp.size()), dim3(64), 0, c.stream, dg.p, k, kMT / (16 >> k),
                       c.d_rastile[k].p);
    PSOCI_HIP(hipGetLastError());
  }
  c.sync();
}

// the plan's tables as the kernels read them
static void ras_upload_view(Ctx& c) {
  RasView v = ras_host_view(c.ras);
  v.mask = c.d_rasmask.p;
  v.cls = c.d_rascls.p;
  v.add = c.d_rasadd.p;
  v.rem = c.d_rasrem.p;
  v.blk = c.d_rasblk.p;
  v.qlist = c.d_rasq.p;
  v.cmp = c.d_rascmp.p;
  v.wunit = c.ras.cwunit;
  v.pidx = c.d_raspidx.p;
  v.sef = c.d_rassef.p;
  c.d_rasview.upload(&v, 1, c.stream);
  c.sync();
}

// Builds the plan's strings: the tables, the SEFs' determinants and the
// determinant vectors, which the adjoint works on as well as the sigma; false
// (c.ras_why says why) when the space does not qualify.
static bool make_strings(Ctx& c, bool adjoint) {
  const Space& sp = c.sp;
  std::vector<double> one(c.d_one.n), two(c.d_two.n);
  c.d_one.download(one.data(), one.size(), c.stream);
  c.d_two.download(two.data(), two.size(), c.stream);
  c.sync();
  // engine 2 on request takes complete EVEN-class spaces only; the automatic
  // choice also odd electron counts and parts of a space, where that is
  // cheaper than the pair records
  ras_plan(c.ras, sp, one.data(), two.data(), c.direct_engine_req == 0);
  if (!c.ras.ok) {
    c.ras_why = c.ras.why;
    return false;
  }
  const RasPlan& P = c.ras;
  {
    DevBuf<int> flag;
    flag.alloc(1);
    PSOCI_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), c.stream));
    hipLaunchKernelGGL(k_ras_zero_singles, dim3(nblk(sp.ncfg * sp.nbf, 256)), dim3(256), 0, c.stream, sp.ncfg,
                       c.d_dm.p, c.d_sm.p, P.emask, P.m, sp.nbf, P.fill < 1.0 ? 0 : 1, c.d_one.p, c.d_two.p, flag.p);
    PSOCI_HIP(hipGetLastError());
    int f = 0;
    flag.download(&f, 1, c.stream);
    c.sync();
    // the string-driven adjoint has no pairs that the reference leaves out
    // (a double excitation both of whose integrals are exactly zero, a single
    // one whose sum is)
    c.ras_rdm = !(f & 2) && !c.zero_integral;
    if (f & 1) {
      c.ras_rdm = false;
      c.ras_why = "a configuration pair one electron apart has vnt[0] exactly zero with nonzero exchange terms";
      c.ras = RasPlan();
      return false;
    }
    if (adjoint && !c.ras_rdm) {
      c.strings_tried = false;  // they may still serve the sigma
      c.ras = RasPlan();
      return false;
    }
  }
  // determinant vectors of 16 FP64 columns where they take a small part of the
  // free memory, else of 16 FP32 or 8 FP64 columns
  {
    size_t fr = 0, tot = 0;
    c.spare.give_back();
    PSOCI_HIP(hipMemGetInfo(&fr, &tot));
    const double rows = 2.0 * (double)P.ndet + 2.0;
    c.ras_kc64 = rows * 128 <= 0.2 * (double)fr ? 16 : 8;
    if (c.ras_kc64 == 8 && rows * 64 > 0.6 * (double)fr) {
      c.ras_why = "needs " + std::to_string((int64_t)(rows * 64 / 1e9)) + " GB of device memory, " +
                  std::to_string((int64_t)(fr / 1000000000)) + " GB free";
      c.strings_tried = !adjoint;
      c.ras = RasPlan();
      return false;
    }
    c.d_rasc.alloc((size_t)(2 * P.ndet + 2) * 8 * c.ras_kc64);
  }
  c.d_rasmask.upload(P.mask, c.stream);
  c.d_rascls.upload(P.cls, c.stream);
  c.d_rasadd.upload(P.add, c.stream);
  c.d_rasrem.upload(P.rem, c.stream);
  c.d_rasblk.upload(P.blk, c.stream);
  c.d_rasq.upload(P.qlist, c.stream);
  c.d_raspidx.upload(P.pidx, c.stream);
  c.d_rassef.upload(P.sef, c.stream);
  ras_upload_view(c);
  // the SEF order
  {
    const int64_t nsef = (int64_t)P.sef.size();
    DevBuf<int64_t> flag, rank;
    DevBuf<int32_t> sef;
    flag.alloc(P.ndet + 1);
    rank.alloc(P.ndet + 1);
    sef.alloc(P.ndet);
    c.d_rasorder.alloc(nsef);
    hipLaunchKernelGGL(k_ras_fill64, dim3(nblk(P.ndet + 1, 256)), dim3(256), 0, c.stream, P.ndet + 1, flag.p,
                       (int64_t)0);
    PSOCI_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_ras_mark, dim3(nblk(nsef, 256)), dim3(256), 0, c.stream, c.d_rasview.p, flag.p, sef.p);
    PSOCI_HIP(hipGetLastError());
    c.scan(flag.p, rank.p, P.ndet + 1);
    int64_t found = 0;
    PSOCI_HIP(hipMemcpyAsync(&found, rank.p + P.ndet, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
    c.sync();
    PSOCI_CHECK(found == nsef, PSOCI_ERR_STATE, "string-driven sigma: inconsistent determinant map");
    hipLaunchKernelGGL(k_ras_order, dim3(nblk(P.ndet, 256)), dim3(256), 0, c.stream, P.ndet, flag.p, rank.p, sef.p,
                       c.d_rasorder.p);
    PSOCI_HIP(hipGetLastError());
    c.sync();
  }
  // the determinants of no SEF
  c.d_rasabsent.release();
  if (P.fill < 1.0) {
    DevBuf<int64_t> absent, rank;
    absent.alloc(P.ndet + 1);
    rank.alloc(P.ndet + 1);
    const int64_t nsef = (int64_t)P.sef.size();
    hipLaunchKernelGGL(k_ras_fill64, dim3(nblk(P.ndet, 256)), dim3(256), 0, c.stream, P.ndet, absent.p, (int64_t)1);
    hipLaunchKernelGGL(k_ras_fill64, dim3(1), dim3(256), 0, c.stream, (int64_t)1, absent.p + P.ndet, (int64_t)0);
    hipLaunchKernelGGL(k_ras_present, dim3(nblk(nsef, 256)), dim3(256), 0, c.stream, c.d_rasview.p, absent.p);
    PSOCI_HIP(hipGetLastError());
    c.scan(absent.p, rank.p, P.ndet + 1);
    int64_t na = 0;
    PSOCI_HIP(hipMemcpyAsync(&na, rank.p + P.ndet, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
    c.sync();
    c.d_rasabsent.alloc(na);
    hipLaunchKernelGGL(k_ras_absent, dim3(nblk(P.ndet, 256)), dim3(256), 0, c.stream, P.ndet, absent.p, rank.p,
                       c.d_rasabsent.p);
    PSOCI_HIP(hipGetLastError());
    c.sync();
  }
  // their determinants' signed rows
  {
    const int64_t nsef = (int64_t)P.sef.size();
    c.d_rasrows.alloc(nsef);
    hipLaunchKernelGGL(k_ras_sefrows, dim3(nblk(nsef, 256)), dim3(256), 0, c.stream, c.d_rasview.p,
                       c.d_rasorder.p, c.d_rasrows.p);
    PSOCI_HIP(hipGetLastError());
    c.sync();
  }
  return true;
}

bool build_strings(Ctx& c, bool adjoint) {
  if (c.strings_tried) return c.have_strings;
  c.strings_tried = true;
  try {
    c.have_strings = make_strings(c, adjoint);
  } catch (...) {
    c.drop_plan();
    c.strings_tried = !adjoint;  // a density's shortage of memory is not the sigma's
    throw;
  }
  return c.have_strings;
}

// The products of the plan: the compact layouts' matrices, the D entries' and
// terms' tables, and W.
static bool make_products(Ctx& c) {
  const RasPlan& P = c.ras;
  if (c.direct_engine_req == 2 && (P.frac || P.fill < 1.0)) {
    c.ras_why = P.frac ? "odd electron count (one determinant per SEF)" : "not a complete RAS configuration space";
    return false;
  }
  {
    // device memory: W and the determinant vectors (16 FP32 / 8 or 16 FP64
    // columns), the term lists; leave room for the caller's vectors
    int64_t terms = 0;
    for (const RasSef& e : P.sef)
      for (int d = 0; d < e.n; ++d) {
        const RasSectorDev& S = P.sec[e.sec[d]];
        terms += (int64_t)S.na * S.nb + (int64_t)S.na * (S.na - 1) / 2 + (int64_t)S.nb * (S.nb - 1) / 2;
      }
    auto needs = [&] {
      return (double)P.cwunit * 64 + (double)P.cdunit * 4 + (double)P.cgunit * 12 + (double)P.ndet * 128 +
             (double)terms * 4 + (double)P.sef.size() * 9;
    };
    size_t fr = 0, tot = 0;
    c.spare.give_back();
    PSOCI_HIP(hipMemGetInfo(&fr, &tot));
    fr += c.d_rasc.n;  // counted below
    // the matrices per row group can take more than the W elements they save
    // (10 + 24 orbitals: 18.8 GB against 17 GB): where that is too much, one
    // matrix per product
    // (that of the full layouts, if its W offsets fit)
    if (needs() > 0.6 * (double)fr && P.wunit < kRasMaxW) ras_compact(c.ras, true);
    const double need = needs();
    // FP64 in chunks of 16 columns (whole 128-byte W and c pieces) when W and
    // c fit twice over in 60 % of the free memory, else chunks of 8
    c.ras_kc64 = need + (double)P.cwunit * 64 + (double)P.ndet * 128 <= 0.6 * (double)fr ? 16 : 8;
    if (need > 0.6 * (double)fr) {
      c.ras_why = "needs " + std::to_string((int64_t)(need / 1e9)) + " GB of device memory, " +
                  std::to_string((int64_t)(fr / 1000000000)) + " GB free";
      c.drop_plan();
      return false;
    }
  }
  c.d_rascmp.upload(P.cmp, c.stream);
  ras_upload_view(c);
  // determinant vectors and W: 16 FP32 or ras_kc64 FP64 columns per chunk
  c.d_rasc.alloc((size_t)(2 * P.ndet + 2) * 8 * c.ras_kc64);
  // the compact products' matrices and the D entries' signed rows
  c.d_rasg64.alloc(P.cgunit);
  c.d_rasg32.alloc(P.cgunit);
  c.d_rasdidx.alloc(P.cdunit);
  {
    DevBuf<double> full;
    full.upload(P.G, c.stream);
    int64_t most = 0;
    for (const RasCmp& C : P.cmp) most = std::max(most, C.nvar * C.nqp);
    DevBuf<int16_t> pr, pos;
    pr.alloc(most);
    pos.alloc(most);
    for (int bi = 0; bi < (int)P.cmp.size(); ++bi) {
      const RasCmp& C = P.cmp[bi];
      if (C.nq == 0) continue;
      hipLaunchKernelGGL(k_ras_pairs, dim3(nblk(C.nvar, 64)), dim3(64), 0, c.stream, c.d_rasview.p, bi, pr.p, pos.p);
      PSOCI_HIP(hipGetLastError());
      const int64_t ng = C.nvar * C.nqp * C.nqp;
      hipLaunchKernelGGL(k_ras_gvar, dim3((unsigned)std::min<int64_t>((ng + 255) / 256, kGvarGrid)), dim3(256), 0,
                         c.stream, C.gbase, ng, C.nqp, P.blk[bi].nqp, pos.p, full.p + P.blk[bi].goff, c.d_rasg64.p,
                         c.d_rasg32.p);
      PSOCI_HIP(hipGetLastError());
      hipLaunchKernelGGL(k_ras_didx, dim3(nblk(C.nrows * C.nqp, 256)), dim3(256), 0, c.stream, c.d_rasview.p, bi, pr.p,
                         c.d_rasdidx.p);
      PSOCI_HIP(hipGetLastError());
    }
    ras_tile_tables(c);
    c.sync();
  }
  // the SEF term lists (merged where an SEF's two determinants read the
  // same W elements): count, scan, fill
  {
    const int64_t nsef = (int64_t)P.sef.size();
    DevBuf<int64_t> cnt;
    cnt.alloc(nsef + 1);
    DevBuf<int> bad;
    bad.alloc(1);
    PSOCI_HIP(hipMemsetAsync(bad.p, 0, sizeof(int), c.stream));
    PSOCI_HIP(hipMemsetAsync(cnt.p + nsef, 0, sizeof(int64_t), c.stream));
    hipLaunchKernelGGL(k_ras_terms<false>, dim3(nblk(nsef, 256)), dim3(256), 0, c.stream, c.d_rasview.p,
                       c.d_rasorder.p, cnt.p, nullptr, nullptr, nullptr, bad.p);
    PSOCI_HIP(hipGetLastError());
    c.d_rastoff.alloc(nsef + 1);
    c.scan(cnt.p, c.d_rastoff.p, nsef + 1);
    int64_t nterm = 0;
    PSOCI_HIP(hipMemcpyAsync(&nterm, c.d_rastoff.p + nsef, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
    c.sync();
    c.d_rasterm.alloc(nterm);
    c.d_rasscl.alloc(nsef);
    hipLaunchKernelGGL(k_ras_terms<true>, dim3(nblk(nsef, 256)), dim3(256), 0, c.stream, c.d_rasview.p,
                       c.d_rasorder.p, nullptr, c.d_rastoff.p, c.d_rasterm.p, c.d_rasscl.p, bad.p);
    PSOCI_HIP(hipGetLastError());
    int b = 0;
    bad.download(&b, 1, c.stream);
    c.sync();
    PSOCI_CHECK(!b, PSOCI_ERR_STATE, "string-driven sigma: inconsistent term lists");
    c.ras_nterm = nterm;
  }
  c.d_rasw.alloc((size_t)P.cwunit * 8 * c.ras_kc64);
  c.sync();
  return true;
}

bool build_ras(Ctx& c) {
  c.ras_tried = true;
  if (!build_strings(c, false)) return false;
  try {
    c.have_ras = make_products(c);
  } catch (...) {
    c.drop_plan();
    throw;
  }
  return c.have_ras;
}

void build_direct(Ctx& c) {
  if (c.direct_engine_req != 1 && !c.have_ras && !c.ras_tried) try {
      if (build_ras(c)) return;
    } catch (const Error& e) {
      // (the pair records may take less)
      if (e.code != PSOCI_ERR_NOMEM || c.direct_engine_req == 2) throw;
    }
  PSOCI_CHECK(c.direct_engine_req != 2 || direct_engine(c) == 2, PSOCI_ERR_UNSUPPORTED,
              c.have_ras ? "the string-driven direct sigma on request takes complete EVEN-class spaces only"
                         : "the string-driven direct sigma does not apply to this space: " + c.ras_why);
  if (!direct_engine(c)) build_pairs(c);
}

void ras_timing(Ctx& c, int prec, int k, int reps, double* ms, double* flops) {
  PSOCI_CHECK(c.have_ras, PSOCI_ERR_STATE, "the string-driven direct sigma is not set up");
  PSOCI_CHECK(k >= 1 && reps >= 1, PSOCI_ERR_ARG, "k and reps must be positive");
  const int64_t n = c.sp.nsef_total;
  const size_t es = prec == PSOCI_FP32 ? 4 : 8;
  DevBuf<char> X, Y;
  X.alloc((size_t)n * k * es);
  Y.alloc((size_t)n * k * es);
  PSOCI_HIP(hipMemsetAsync(X.p, 0, (size_t)n * k * es, c.stream));
  double acc[5] = {0, 0, 0, 0, 0};
  for (int r = 0; r < reps; ++r) {
    RasTiming tm;
    if (prec == PSOCI_FP32)
      ras_any_k<float>(c, k, reinterpret_cast<const float*>(X.p), k, reinterpret_cast<float*>(Y.p), k, &tm);
    else
      ras_any_k<double>(c, k, reinterpret_cast<const double*>(X.p), k, reinterpret_cast<double*>(Y.p), k, &tm);
    PSOCI_HIP(hipEventSynchronize(tm.ev.back()));
    for (size_t i = 0; i < tm.group.size(); ++i) {
      float t = 0.f;
      PSOCI_HIP(hipEventElapsedTime(&t, tm.ev[i], tm.ev[i + 1]));
      acc[tm.group[i]] += t;
    }
  }
  for (int g = 0; g < 5; ++g) ms[g] = acc[g] / reps;
  if (flops) {
    for (int g = 0; g < 3; ++g) flops[g] = 0.0;
    for (const RasCmp& C : c.ras.cmp) flops[C.kind] += 2.0 * (double)C.nrows * C.nq * C.nq * k;
  }
}

int ras_scatter64(Ctx& c, const double* X, int ldx, int col0, int kw) {
  const int64_t nsef = (int64_t)c.ras.sef.size();
  double* cv = reinterpret_cast<double*>(c.d_rasc.p);
  const int kc = ras_width64(kw);
  const dim3 grid(8 * nblk(nsef * kc, 8 * 256));
  const int64_t na = (int64_t)c.d_rasabsent.n;
  switch (kc) {
#define PSOCI_RAS_SCATTER(KCV)                                                                                   \
  case KCV:                                                                                                      \
    hipLaunchKernelGGL((k_ras_x2c<double, KCV, double>), grid, dim3(256), 0, c.stream, nsef, c.ras.ndet,         \
                       c.d_rasorder.p, c.d_rasrows.p, X, ldx, col0, kw, cv);                                     \
    if (na)                                                                                                      \
      hipLaunchKernelGGL((k_ras_blank<double, KCV>), dim3(nblk(na * KCV, 256)), dim3(256), 0, c.stream, na,      \
                         c.ras.ndet, c.d_rasabsent.p, cv);                                                       \
    break;
    PSOCI_RAS_SCATTER(16)
    PSOCI_RAS_SCATTER(8)
    PSOCI_RAS_SCATTER(4)
    PSOCI_RAS_SCATTER(2)
#undef PSOCI_RAS_SCATTER
  }
  PSOCI_HIP(hipGetLastError());
  return kc;
}

void sigma_ras(Ctx& c, int prec, int k, const void* X, int ldx, void* Y, int ldy) {
  PSOCI_CHECK(c.have_ras, PSOCI_ERR_STATE, "the string-driven direct sigma is not set up");
  if (prec == PSOCI_FP32)
    ras_any_k<float>(c, k, static_cast<const float*>(X), ldx, static_cast<float*>(Y), ldy);
  else
    ras_any_k<double>(c, k, static_cast<const double*>(X), ldx, static_cast<double*>(Y), ldy);
}

}  // namespace psoci
