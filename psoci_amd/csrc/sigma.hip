// Sigma (H . X for k vectors) from the stored Hamiltonian.
//
// Replaces matrixVectorProductsSplitChunkMultipleJchunks
// (PsociGAhamiltonian.C:6921-7269), which forms y_i += sum_j H_ij x_j and
// y_j += H_ij x_i from the stored lower triangle, one vector at a time, with
// per-row GA gets and an all-reduce of y per chunk.  Here H is resident in
// HBM as the symmetric full CSR (lower part of each row first), X and Y are
// [n][k] row-major (the reference's GA vector layout), and one wavefront
// reduces one row for all k vectors at once: the row's values and columns
// stream from HBM once per launch, X rows are gathered from L2/MALL.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

#include "ctx.hpp"
#include "pad.hpp"

namespace psoci {

namespace {

constexpr int kWave = 64;

template <typename T>
__device__ __forceinline__ T fmadd(T a, T b, T c);
template <>
__device__ __forceinline__ double fmadd<double>(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}
template <>
__device__ __forceinline__ float fmadd<float>(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}

template <typename T, int N>
struct PieceOf {
  typedef T type __attribute__((ext_vector_type(N)));
  typedef T loose __attribute__((ext_vector_type(N), aligned(sizeof(T))));  // any start of a row
};

// the value that lane g of this lane's group of G holds (G = 1, 2, 4: groups
// lie within quads, one DPP move per 32 bits)
template <int G, int g>
__device__ __forceinline__ int32_t of_lane(int32_t x) {
  if constexpr (G == 1) return x;
  constexpr int ctrl = G == 2 ? (g | g << 2 | (2 + g) << 4 | (2 + g) << 6) : (g | g << 2 | g << 4 | g << 6);
  return __builtin_amdgcn_mov_dpp(x, ctrl, 0xf, 0xf, true);
}
template <int G, int g>
__device__ __forceinline__ float of_lane(float x) {
  return __int_as_float(of_lane<G, g>(__float_as_int(x)));
}
template <int G, int g>
__device__ __forceinline__ double of_lane(double x) {
  return __hiloint2double(of_lane<G, g>(__double2hiint(x)), of_lane<G, g>(__double2loint(x)));
}

// R rows per wavefront (64/R lanes per row: short rows share a wavefront)
// and G lanes per nonzero (each of them multiplies K/G of the K columns, so
// the G lanes of a nonzero read one contiguous piece of its x row).  In a
// turn every lane of a row loads the columns and values of U consecutive
// nonzeros (16-byte loads, one turn ahead), and the groups of G lanes walk
// their G U nonzeros, each taken from the lane that holds it.  Four (two at 64
// bytes of x per lane) accumulators per column, so that the chains are no
// longer than with one row per wavefront.  Partial sums are reduced across the
// groups of the row with shuffles.  rows (optional): the launch covers the
// nrows rows listed there (one row-length bucket) instead of 0..n-1.
// Bound by the matrix stream and the x gathers from L2 (a 64-byte row piece
// per nonzero).  31,650 rows of 715 nonzeros (10 orbitals, 8 electrons), each
// call on another matrix than the last: FP32 16 columns 169 -> 125 us, FP64 4
// / 16 columns 200 -> 114 / 218 -> 185 us against lanes that loaded every
// nonzero of their group themselves, one at a time.
template <typename T, int K, int G, int R>
__global__ __launch_bounds__(256) void k_spmm(int64_t nrows, const int32_t* __restrict__ rows,
                                              const int64_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                              const T* __restrict__ val, const T* __restrict__ X, int ldx,
                                              T* __restrict__ Y, int ldy) {
  constexpr int LR = kWave / R;   // lanes per row
  constexpr int C = K / G;        // columns per lane
  constexpr int U = 8;            // nonzeros a lane loads per turn
  constexpr int XB = C * sizeof(T) >= 64 ? 4 : 8;  // of which so many x pieces are in flight
  constexpr int PW = C * sizeof(T) % 16 == 0 ? 16 / sizeof(T) : 1;  // values per x load
  constexpr int NA = C * sizeof(T) <= 32 ? 4 : 2;                   // accumulators per column
  constexpr int VW = 16 / sizeof(T);                                // values per load
  typedef typename PieceOf<T, PW>::type V;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t slot_r =
      ((int64_t)blockIdx.x * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave)) * R + lane / LR;
  const bool live = slot_r < nrows;
  const int64_t r = live ? (rows ? (int64_t)rows[slot_r] : slot_r) : 0;
  const int lr = lane % LR, cc = lr % G;
  T acc[NA][C];
#pragma unroll
  for (int x = 0; x < NA; ++x)
#pragma unroll
    for (int v = 0; v < C; ++v) acc[x][v] = (T)0;
  const int64_t lo = live ? rowptr[r] : 0;
  const int len = live ? (int)(rowptr[r + 1] - lo) : 0;
  const T* __restrict__ vr = val + lo;
  const int32_t* __restrict__ cr = col + lo;
  const T* __restrict__ xc = X + cc * C;
  // this lane's nonzeros of a turn; past the row's end the row's last one,
  // its column complemented: left out of the sums
  T a[U];
  int32_t j[U];
  auto fetch = [&](int q) {
    if (q + U <= len) {
#pragma unroll
      for (int u = 0; u < U; u += VW) {
        const auto t = *reinterpret_cast<const typename PieceOf<T, VW>::loose*>(vr + q + u);
#pragma unroll
        for (int i = 0; i < VW; ++i) a[u + i] = t[i];
      }
#pragma unroll
      for (int u = 0; u < U; u += 4) {
        const auto t = *reinterpret_cast<const typename PieceOf<int32_t, 4>::loose*>(cr + q + u);
#pragma unroll
        for (int i = 0; i < 4; ++i) j[u + i] = t[i];
      }
    } else if (len > 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = q + u < len ? q + u : len - 1;
        a[u] = vr[t];
        j[u] = q + u < len ? cr[t] : ~cr[t];
      }
    }
  };
  const int q = lr * U;  // this lane's first nonzero of the turn
  int base = 0;
  if (len > 0) fetch(q);
  while (base < len) {
    T b[U];
    int32_t jj[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      b[u] = a[u];
      jj[u] = j[u];
    }
    base += LR * U;
    if (base < len) fetch(q + base);
    auto sub = [&](auto gc) {
      constexpr int g = decltype(gc)::value;
#pragma unroll
      for (int h = 0; h < U; h += XB) {
        V xv[XB][C / PW];
        T w[XB];
        int32_t c[XB];
#pragma unroll
        for (int u = 0; u < XB; ++u) {
          c[u] = of_lane<G, g>(jj[h + u]);
          w[u] = of_lane<G, g>(b[h + u]);
          const V* x = reinterpret_cast<const V*>(xc + (int64_t)(c[u] < 0 ? ~c[u] : c[u]) * ldx);
#pragma unroll
          for (int p = 0; p < C / PW; ++p) xv[u][p] = x[p];
        }
#pragma unroll
        for (int u = 0; u < XB; ++u)
#pragma unroll
          for (int v = 0; v < C; ++v) {
            const T f = fmadd(w[u], xv[u][v / PW][v % PW], acc[u % NA][v]);
            acc[u % NA][v] = c[u] < 0 ? acc[u % NA][v] : f;
          }
      }
    };
    sub(std::integral_constant<int, 0>{});
    if constexpr (G >= 2) sub(std::integral_constant<int, 1>{});
    if constexpr (G >= 4) {
      sub(std::integral_constant<int, 2>{});
      sub(std::integral_constant<int, 3>{});
    }
  }
  T sum[C];
#pragma unroll
  for (int v = 0; v < C; ++v) {
    sum[v] = acc[0][v] + acc[1][v];
    if constexpr (NA == 4) sum[v] += acc[2][v] + acc[3][v];
  }
  // reduce over the groups of the row (lane bits G .. LR-1)
#pragma unroll
  for (int off = G; off < LR; off <<= 1) {
#pragma unroll
    for (int v = 0; v < C; ++v) sum[v] += __shfl_xor(sum[v], off, kWave);
  }
  if (live && lr < G) {
    T* y = Y + r * ldy + cc * C;
#pragma unroll
    for (int v = 0; v < C; ++v) y[v] = sum[v];
  }
}

template <typename T, int K, int G, int R>
void launch_gr(Ctx& c, const T* val, const T* X, int ldx, T* Y, int ldy, const int32_t* rows, int64_t nrows) {
  const int64_t rows_per_block = 4 * R;
  if (nrows <= 0) return;
  hipLaunchKernelGGL((k_spmm<T, K, G, R>), dim3((unsigned)((nrows + rows_per_block - 1) / rows_per_block)), dim3(256),
                     0, c.stream, nrows, rows, c.d_rowptr.p, c.d_col.p, val, X, ldx, Y, ldy);
  PSOCI_HIP(hipGetLastError());
}

// one launch of shape (g lanes per nonzero, r rows per wavefront) over the
// listed rows (rows null: all n)
template <typename T, int K>
void launch_shape(Ctx& c, int g0, int r, const T* val, const T* X, int ldx, T* Y, int ldy, const int32_t* rows,
                  int64_t nrows) {
  const int g = K >= g0 ? g0 : 1;
  const int key = g * 16 + r;
  switch (key) {
#define PSOCI_SPMM_CASE(GG, RR)                                                    \
  case GG * 16 + RR:                                                               \
    if constexpr (K >= GG) {                                                       \
      launch_gr<T, K, (K >= GG ? GG : 1), RR>(c, val, X, ldx, Y, ldy, rows, nrows); \
      return;                                                                      \
    }                                                                              \
    break;
    PSOCI_SPMM_CASE(1, 1)
    PSOCI_SPMM_CASE(1, 2)
    PSOCI_SPMM_CASE(1, 4)
    PSOCI_SPMM_CASE(1, 8)
    PSOCI_SPMM_CASE(2, 1)
    PSOCI_SPMM_CASE(2, 2)
    PSOCI_SPMM_CASE(2, 4)
    PSOCI_SPMM_CASE(2, 8)
    PSOCI_SPMM_CASE(4, 1)
    PSOCI_SPMM_CASE(4, 2)
    PSOCI_SPMM_CASE(4, 4)
    PSOCI_SPMM_CASE(4, 8)
#undef PSOCI_SPMM_CASE
    default: break;
  }
  launch_gr<T, K, 1, 1>(c, val, X, ldx, Y, ldy, rows, nrows);
}

// Shape rule of a launch of K columns: each lane reads 16 bytes of an x row
// (G = K sizeof / 16 lanes, at most 4).  More rows per wavefront waste less of a
// row's last turn and of its reduction (gain), if there are wavefronts enough
// to hide the loads behind; fewer spread the rows more evenly over the compute
// units.  FP32 sums of G = 4 take at most four rows, whose chains are no longer
// than those of one lane per nonzero.  us per call over R = 1, 2, 4, 8:
//   rows (nonzeros each)   FP32 1 column            FP64 16 columns
//   2,044 (266)            18.2 18.5 19.4 20.1      22.5 22.9 24.4 28.7
//   9,080 (870)            32.0 32.6 33.8 35.6      62.8 66.9 73.4 88.4
//   18,354 (650, uneven)   43.4 42.3 43.6 45.2       106   97   99  127
//   31,650 (715)           64.5 65.1 60.9 54.8       190  186  179  170
//   122,235 (3,508)        1301 1203 1076  946      3802 3309 3155 2826
//   257,670 (5,179)        4227 3915 3466 3014     13161 11555 10845 9278
// and over K on 31,650 rows: FP32 1 / 4 / 8 / 16 / 32 columns 55 / 68 / 81 / 106
// / 152, FP64 81 / 105 / 125 / 169 against one lane per nonzero at its best R
// 55 / 68 / 103 / 175 / 397, 85 / 125 / 193 / 392.
struct SpmmShape {
  int g, r;
};
inline SpmmShape spmm_shape(size_t es, int K, int64_t rows, int units) {
  SpmmShape s;
  s.g = std::max(1, std::min(4, (int)(K * es) / 16));
  s.r = 1;
  double best = 0.0;
  for (int r = 1, i = 0; r <= (es == 4 && s.g == 4 ? 4 : 8); r *= 2, ++i) {
    const double gain[4] = {0.0, 0.08, 0.18, 0.30};
    const double load = std::ceil((double)rows / (4 * r)) / units;  // workgroups per unit
    if (r > 1 && load <= 1.0) break;
    const double score = load / std::ceil(load) * (1.0 + gain[i] * std::min(1.0, (load - 1.0) / 3.0));
    if (score > best) {
      best = score;
      s.r = r;
    }
  }
  return s;
}

// one launch over all rows, or one per non-empty row-length bucket; the
// rule's shape, or the fixed one
template <typename T, int K>
void launch_spmm(Ctx& c, const T* val, const T* X, int ldx, T* Y, int ldy) {
  const int pi = sizeof(T) == 4 ? 1 : 0;
  if (!c.spmm_bucketed[pi]) {
    const int64_t n = c.sp.nsef_total;
    SpmmShape s = spmm_shape(sizeof(T), K, n, c.units);
    if (c.spmm_fixed[pi]) s = {c.spmm_g[pi], c.spmm_r[pi]};
    launch_shape<T, K>(c, s.g, s.r, val, X, ldx, Y, ldy, nullptr, n);
    return;
  }
  for (int b = 0; b < kSpmmBuckets; ++b) {
    const int64_t lo = c.spmm_boff[b], cnt = c.spmm_boff[b + 1] - lo;
    if (cnt <= 0) continue;
    SpmmShape s = spmm_shape(sizeof(T), K, cnt, c.units);
    if (c.spmm_fixed[pi]) s = {c.spmm_bg[pi][b], c.spmm_br[pi][b]};
    launch_shape<T, K>(c, s.g, s.r, val, X, ldx, Y, ldy, c.d_brows.p + lo, cnt);
  }
}

template <typename T>
void spmm_any_k(Ctx& c, const T* val, int k, const T* X, int ldx, T* Y, int ldy, const Staging& st) {
  pad::blocks<T>(c, c.sp.nsef_total, k, 32, X, ldx, Y, ldy, [&](int K, const T* x, int lx, T* y, int ly) {
    switch (K) {
      case 32:
        // FP64: 32 columns' sums and x pieces leave too few wavefronts (18,354
        // rows: 368 us, 31,650 rows: 459 us, against twice 97 and 170 us)
        if constexpr (sizeof(T) == 8) {
          launch_spmm<T, 16>(c, val, x, lx, y, ly);
          launch_spmm<T, 16>(c, val, x + 16, lx, y + 16, ly);
        } else {
          launch_spmm<T, 32>(c, val, x, lx, y, ly);
        }
        break;
      case 16: launch_spmm<T, 16>(c, val, x, lx, y, ly); break;
      case 8: launch_spmm<T, 8>(c, val, x, lx, y, ly); break;
      case 4: launch_spmm<T, 4>(c, val, x, lx, y, ly); break;
      case 2: launch_spmm<T, 2>(c, val, x, lx, y, ly); break;
      default: launch_spmm<T, 1>(c, val, x, lx, y, ly); break;
    }
  }, false, st);
}

}  // namespace

namespace {
const int64_t kBucketLim[kSpmmBuckets] = {64, 256, 1024, 4096, INT64_MAX};

// rows per row-length class
__global__ __launch_bounds__(256) void k_bucket_count(int64_t n, const int64_t* __restrict__ rowptr,
                                                      unsigned long long* __restrict__ out) {
  __shared__ unsigned long long cnt[kSpmmBuckets];
  if (threadIdx.x < kSpmmBuckets) cnt[threadIdx.x] = 0;
  __syncthreads();
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
    const int64_t len = rowptr[r + 1] - rowptr[r];
    const int b = len < 64 ? 0 : len < 256 ? 1 : len < 1024 ? 2 : len < 4096 ? 3 : 4;
    atomicAdd(&cnt[b], 1ull);
  }
  __syncthreads();
  if (threadIdx.x < kSpmmBuckets && cnt[threadIdx.x]) atomicAdd(&out[threadIdx.x], cnt[threadIdx.x]);
}
__global__ void k_bucket_zero(unsigned long long* out) {
  if (threadIdx.x < kSpmmBuckets) out[threadIdx.x] = 0;
}
}  // namespace

// Row-length buckets of the stored matrix (full symmetric rows): lengths
// < 64, 64-255, 256-1023, 1024-4095, >= 4096; the row lists in ascending
// order per bucket, made when the bucketed launches are used.  A property of
// the matrix alone, so a loaded checkpoint gets the same buckets.
static void count_buckets(Ctx& c) {
  const int64_t n = c.sp.nsef_total;
  DevBuf<unsigned long long> d;
  d.alloc(kSpmmBuckets);
  hipLaunchKernelGGL(k_bucket_zero, dim3(1), dim3(64), 0, c.stream, d.p);
  hipLaunchKernelGGL(k_bucket_count, dim3((unsigned)std::min<int64_t>(256, (n + 255) / 256)), dim3(256), 0, c.stream, n,
                     c.d_rowptr.p, d.p);
  PSOCI_HIP(hipGetLastError());
  unsigned long long h[kSpmmBuckets];
  d.download(h, kSpmmBuckets, c.stream);
  c.sync();
  c.spmm_boff[0] = 0;
  for (int b = 0; b < kSpmmBuckets; ++b) c.spmm_boff[b + 1] = c.spmm_boff[b] + (int64_t)h[b];
}
static void list_buckets(Ctx& c) {
  const int64_t n = c.sp.nsef_total;
  std::vector<int64_t> rp(n + 1);
  c.d_rowptr.download(rp.data(), n + 1, c.stream);
  c.sync();
  std::vector<int32_t> rows;
  rows.reserve(n);
  for (int b = 0; b < kSpmmBuckets; ++b) {
    const int64_t lo = b ? kBucketLim[b - 1] : 0;
    for (int64_t r = 0; r < n; ++r) {
      const int64_t len = rp[r + 1] - rp[r];
      if (len >= lo && len < kBucketLim[b]) rows.push_back((int32_t)r);
    }
  }
  c.d_brows.upload(rows, c.stream);
  c.sync();
}

// The stored sigma's shapes (spmm_shape; those at 16 columns are reported).
// PSOCI_SPMM_SHAPE=<G>x<R> fixes one shape for every width.  All rows go in
// one launch; PSOCI_SPMM_BUCKETS=1 launches them by length class, which took 3
// to 8 % longer on 31,650 to 45,304 rows and 10 to 45 % on 17,022 and 18,354
// (fewer rows per launch), the same on 48,852 and 263,004, and 8 to 17 % less on
// 257,670 rows whose configurations mix two lengths (5,877 and 2,976).  saved (a checkpoint's): its
// fixed shapes and its choice of launches stand for that precision.
void tune_stored(Ctx& c, const SpmmSaved* saved) {
  count_buckets(c);
  const int64_t n = c.sp.nsef_total;
  PSOCI_HIP(hipDeviceGetAttribute(&c.units, hipDeviceAttributeMultiprocessorCount, c.device));
  int eg = 0, er = 0;
  if (const char* env = std::getenv("PSOCI_SPMM_SHAPE")) {
    int g = 1, r = 1;
    if (std::sscanf(env, "%dx%d", &g, &r) == 2 && (g == 1 || g == 2 || g == 4) &&
        (r == 1 || r == 2 || r == 4 || r == 8)) {
      eg = g;
      er = r;
      saved = nullptr;
    }
  }
  for (int pi = 0; pi < 2; ++pi) {
    c.spmm_tune_ms[pi] = c.spmm_bucket_ms[pi] = -1.0;
    if (saved && saved->fixed[pi]) {
      c.spmm_fixed[pi] = true;
      c.spmm_g[pi] = saved->g[pi];
      c.spmm_r[pi] = saved->r[pi];
      c.spmm_bucketed[pi] = saved->bucketed[pi];
      std::copy(saved->bg[pi], saved->bg[pi] + kSpmmBuckets, c.spmm_bg[pi]);
      std::copy(saved->br[pi], saved->br[pi] + kSpmmBuckets, c.spmm_br[pi]);
      continue;
    }
    const size_t es = pi ? 4 : 8;
    const SpmmShape s = spmm_shape(es, 16, n, c.units);
    c.spmm_fixed[pi] = eg != 0;
    c.spmm_g[pi] = eg ? eg : s.g;
    c.spmm_r[pi] = er ? er : s.r;
    int nonempty = 0;
    for (int b = 0; b < kSpmmBuckets; ++b) {
      const int64_t cnt = c.spmm_boff[b + 1] - c.spmm_boff[b];
      c.spmm_bg[pi][b] = eg ? eg : 1;
      c.spmm_br[pi][b] = er ? er : 1;
      if (cnt <= 0) continue;
      ++nonempty;
      const SpmmShape t = spmm_shape(es, 16, cnt, c.units);
      if (!eg) {
        c.spmm_bg[pi][b] = t.g;
        c.spmm_br[pi][b] = t.r;
      }
    }
    c.spmm_bucketed[pi] = false;
    if (const char* eb = std::getenv("PSOCI_SPMM_BUCKETS")) c.spmm_bucketed[pi] = nonempty > 1 && eb[0] == '1';
    if (eg) c.spmm_bucketed[pi] = false;
    if (saved && saved->chosen[pi]) c.spmm_bucketed[pi] = saved->bucketed[pi];
  }
  if (c.spmm_bucketed[0] || c.spmm_bucketed[1]) list_buckets(c);
}

void sigma_stored(Ctx& c, int prec, int k, const void* X, int ldx, void* Y, int ldy, const Staging& st) {
  PSOCI_CHECK(c.have_h, PSOCI_ERR_STATE, "stored sigma needs psoci_build_h first");
  if (prec == PSOCI_FP32)
    spmm_any_k<float>(c, c.d_val32.p, k, static_cast<const float*>(X), ldx, static_cast<float*>(Y), ldy, st);
  else
    spmm_any_k<double>(c, c.d_val.p, k, static_cast<const double*>(X), ldx, static_cast<double*>(Y), ldy, st);
}

size_t sigma_staging_bytes(const Ctx& c, int mode, int prec, int k, const void* X, int ldx, const void* Y, int ldy) {
  // the stored sigma has widths 1..32 (powers of two), the direct one also 24
  const bool w24 = mode == PSOCI_SIGMA_DIRECT;
  const int64_t n = c.sp.nsef_total;
  if (mode == PSOCI_SIGMA_DIRECT && direct_engine(c) == 2) return 0;  // reads X and writes Y at their strides
  if (prec == PSOCI_FP32)
    return pad::staging_bytes<float>(n, k, 32, static_cast<const float*>(X), ldx, static_cast<const float*>(Y), ldy,
                                     w24);
  return pad::staging_bytes<double>(n, k, 32, static_cast<const double*>(X), ldx, static_cast<const double*>(Y), ldy,
                                    w24);
}

}  // namespace psoci
