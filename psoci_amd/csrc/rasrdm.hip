// Adjoint of the energies on the string plan (ras.hpp): for its spaces the
// generalised 1- and 2-RDM that psoci_rdm returns are contractions of Gram
// matrices.
//
// E = sum_k w_k c_k^T H c_k is, per product of the plan (RasBlockDev), the sum
// over its rows of D^T G D with G the product's integral matrix, so
// dE/dG = M = sum over rows and roots of w_k D D^T: a symmetric
// rank-(rows x roots) update on FP64 MFMA (k_ras_gram), summed over the
// blocks that share G, and dE/dtheta the sum of M over the entries of G that
// read theta (k_ras_grad2, k_ras_grad1: a gather per packed integral).  No
// atomics: the results are reproducible.  Replaces, for these spaces, the
// pair walk of rdm.hip, which generates every SEF element and adds to a few
// integrals with atomics: four roots of the 10-orbital, 8-electron full CI
// 22.6 -> 0.43 ms a call, and no pair records (56 ms of set-up) for a gradient.
//
// The pair walk leaves out pairs whose integral sums are exactly zero (the
// reference computes no block for them); the Gram matrices do not, so spaces
// and integrals with such pairs keep the pair walk (Ctx::ras_rdm).
#include <algorithm>

#include "ctx.hpp"
#include "ras.hpp"

namespace psoci {

namespace {

inline unsigned nblk(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int kPT = 64;       // pairs per tile of M
constexpr int kKK = 16;       // (row, root) values per LDS chunk
constexpr int kLd = kPT + 16; // LDS row stride: the four rows an operand read touches in separate banks

// One tile (ti >= tj) of a block's M over one range of its rows, written to
// its own place (part).  256 threads: thread t stages pair t % 64, values 4
// (t / 64) .. + 3 of a chunk (rows row0 + 4 (t / 64) / KC, roots), so the row
// and its strings are uniform over a wavefront; the next chunk's values are
// loaded while the current one multiplies.  Four wavefronts of 32 x 32.
// Bound by the chain string table -> determinant row of a chunk, so many
// workgroups per CU (20 KB of LDS) and not by the FP64 matrix pipe.
template <int KC>
__global__ __launch_bounds__(256) void k_ras_gram(const RasView* __restrict__ vp, int bi, double fac,
                                                  const double* __restrict__ c, const double* __restrict__ wk,
                                                  int64_t rows_per, double* __restrict__ part) {
  const RasView& v = *vp;
  const RasBlockDev& B = v.blk[bi];
  __shared__ double As[kKK][kLd], Bs[kKK][kLd];
  int ti = 0, tj = (int)blockIdx.x;
  while (tj > ti) tj -= ++ti;  // tile pair blockIdx.x of the lower triangle
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t r0 = (int64_t)blockIdx.y * rows_per;
  const int64_t r1 = r0 + rows_per < B.nrows ? r0 + rows_per : B.nrows;
  constexpr int RC = kKK / KC;              // rows per chunk
  constexpr int NE = KC >= 4 ? 1 : 4 / KC;  // D entries per thread and tile
  const int col = (4 * wave) % KC;
  const int ja = ti * kPT + lane, jb = tj * kPT + lane;
  const int pa = ja < B.nq ? v.qlist[B.qoff + ja] : -1, pb = jb < B.nq ? v.qlist[B.qoff + jb] : -1;
  double wv[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) wv[x] = wk[(col + x) % KC];

  double av[4], bv[4];
  auto load = [&](int64_t rc) {
#pragma unroll
    for (int x = 0; x < 4; ++x) av[x] = bv[x] = 0.0;
#pragma unroll
    for (int n = 0; n < NE; ++n) {
      const int64_t row = rc + (KC >= 4 ? (4 * wave) / KC : NE * wave + n);
      if (row >= r1) continue;
      int64_t u, w;
      double f = fac;
      if (B.tri) {
        ras_tri_uw(row, B.nu, u, w);
        if (u == w) f *= 0.5;  // u < w stands for (w, u) too
      } else {
        u = row / B.nw;
        w = row % B.nw;
      }
      constexpr int NV = KC >= 4 ? 4 : KC;
      if (pa >= 0) {
        int neg = 0;
        const int64_t d = ras_d_det(v, B.kind, B.sector, B.lu, B.lw, B.u0 + u, B.w0 + w, pa & 0xff, (pa >> 8) & 0xff, neg);
        if (d >= 0 && d < v.ndet) {
          const double* __restrict__ src = c + (d + neg * v.ndet) * KC + (KC >= 4 ? col : 0);
#pragma unroll
          for (int x = 0; x < NV; ++x) av[n * NV + x] = f * wv[n * NV + x] * src[x];
        }
      }
      if (pb >= 0) {
        int neg = 0;
        const int64_t d = ras_d_det(v, B.kind, B.sector, B.lu, B.lw, B.u0 + u, B.w0 + w, pb & 0xff, (pb >> 8) & 0xff, neg);
        if (d >= 0 && d < v.ndet) {
          const double* __restrict__ src = c + (d + neg * v.ndet) * KC + (KC >= 4 ? col : 0);
#pragma unroll
          for (int x = 0; x < NV; ++x) bv[n * NV + x] = src[x];
        }
      }
    }
  };
  v4d acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = v4d{0, 0, 0, 0};
  const int kr = lane >> 4, l15 = lane & 15;
  load(r0);
  for (int64_t rc = r0; rc < r1; rc += RC) {
    __syncthreads();  // the chunk before has been read
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      As[4 * wave + x][lane] = av[x];
      Bs[4 * wave + x][lane] = bv[x];
    }
    __syncthreads();
    if (rc + RC < r1) load(rc + RC);
#pragma unroll
    for (int kk = 0; kk < kKK / 4; ++kk) {
      double a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = As[4 * kk + kr][32 * (wave >> 1) + 16 * i + l15];
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = Bs[4 * kk + kr][32 * (wave & 1) + 16 * j + l15];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }
  double* __restrict__ out = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * kPT * kPT;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        out[(32 * (wave >> 1) + 16 * i + 4 * t + kr) * kPT + 32 * (wave & 1) + 16 * j + l15] = acc[i][j][t];
}

// M[i][j] (i >= j tiles; ld nq) += the sum of the row ranges' tiles, in order
__global__ __launch_bounds__(256) void k_ras_gram_sum(int ntp, int nsplit, const double* __restrict__ part, int nq,
                                                      double* __restrict__ M) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)ntp * kPT * kPT) return;
  int ti = 0, tj = (int)(e / (kPT * kPT));
  while (tj > ti) tj -= ++ti;
  const int i = ti * kPT + (int)(e / kPT % kPT), j = tj * kPT + (int)(e % kPT);
  if (i >= nq || j >= nq) return;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  const int64_t st = (int64_t)ntp * kPT * kPT;
  int x = 0;
  for (; x + 4 <= nsplit; x += 4)
#pragma unroll
    for (int y = 0; y < 4; ++y) s[y] += part[e + (x + y) * st];
  for (; x < nsplit; ++x) s[0] += part[e + x * st];
  M[(int64_t)i * nq + j] += (s[0] + s[1]) + (s[2] + s[3]);
}

__global__ __launch_bounds__(256) void k_ras_fill0(int64_t n, double* __restrict__ p) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0.0;
}

__device__ __forceinline__ double gram_at(const RasGradMat& G, const double* __restrict__ M,
                                          const int16_t* __restrict__ px, int nbf, int p, int r, int q, int s) {
  const int i = px[p * nbf + r], j = px[q * nbf + s];
  if (i < 0 || j < 0) return 0.0;
  // tiles above the diagonal are not stored
  return (i / kPT >= j / kPT) ? M[G.moff + (int64_t)i * G.nq + j] : M[G.moff + (int64_t)j * G.nq + i];
}

// dE/d(ij|kl): M over the distinct index orders of the packed integral.  An
// alpha-beta entry [(p,r)][(q,s)] reads (pq|rs); a same-spin one (p > r, q >
// s) reads (pq|rs) - (ps|rq).
__global__ __launch_bounds__(256) void k_ras_grad2(int nbf, int64_t n2, int nmat, const RasGradMat* __restrict__ mat,
                                                   const int16_t* __restrict__ pidx, const double* __restrict__ M,
                                                   double* __restrict__ g2) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n2) return;
  auto split = [](int64_t x, int& hi, int& lo) {
    int a = (int)((sqrt(8.0 * (double)x + 1.0) - 1.0) * 0.5);
    while ((int64_t)a * (a + 1) / 2 > x) --a;
    while ((int64_t)(a + 1) * (a + 2) / 2 <= x) ++a;
    hi = a;
    lo = (int)(x - (int64_t)a * (a + 1) / 2);
  };
  int ij, kl, i, j, k, l;
  split(t, ij, kl);
  split(ij, i, j);
  split(kl, k, l);
  double s = 0.0;
  for (int o = 0; o < 8; ++o) {
    // order o of (ij|kl): bit 0 swaps i j, bit 1 swaps k l, bit 2 the pairs;
    // an order equal to a lower one is left out
    if ((o & 1) && i == j) continue;
    if ((o & 2) && k == l) continue;
    if ((o & 4) && ij == kl) continue;
    int a = (o & 1) ? j : i, b = (o & 1) ? i : j, c = (o & 2) ? l : k, d = (o & 2) ? k : l;
    if (o & 4) {
      int x = a;
      a = c;
      c = x;
      x = b;
      b = d;
      d = x;
    }
    for (int m = 0; m < nmat; ++m) {
      const RasGradMat G = mat[m];
      const int16_t* __restrict__ px = pidx + (int64_t)G.id * nbf * nbf;
      if (G.kind == 0) {
        s += gram_at(G, M, px, nbf, a, c, b, d);
      } else if (a > c) {
        if (b > d) s += gram_at(G, M, px, nbf, a, c, b, d);
        if (d > b) s -= gram_at(G, M, px, nbf, a, c, d, b);
      }
    }
  }
  g2[t] = s;
}

// dE/dh_xy: the one-electron integrals folded into the matrices (ras_plan)
__global__ __launch_bounds__(64) void k_ras_grad1(int nbf, int n1, int nmat, const RasGradMat* __restrict__ mat,
                                                  const int16_t* __restrict__ pidx, const double* __restrict__ M,
                                                  double* __restrict__ g1) {
  const int e = (int)blockIdx.x;
  int hi = 0;
  while ((hi + 1) * (hi + 2) / 2 <= e) ++hi;
  const int lo = e - hi * (hi + 1) / 2;
  if (e >= n1) return;
  double s = 0.0;
  // lane z: the spectator orbital
  for (int z = threadIdx.x; z < nbf; z += 64)
    for (int o = 0; o < (hi == lo ? 1 : 2); ++o) {
      const int x = o ? lo : hi, y = o ? hi : lo;
      for (int m = 0; m < nmat; ++m) {
        const RasGradMat G = mat[m];
        const int16_t* __restrict__ px = pidx + (int64_t)G.id * nbf * nbf;
        if (G.kind == 0) {
          if (G.hr != 0.0) s += G.hr * gram_at(G, M, px, nbf, x, z, y, z);
          if (G.hp != 0.0) s += G.hp * gram_at(G, M, px, nbf, z, x, z, y);
        } else if (G.hr != 0.0) {
          // + h_pq (r = s) + h_rs (p = q) - h_rq (p = s) - h_ps (r = q)
          double d = 0.0;
          if (x > z && y > z) d += gram_at(G, M, px, nbf, x, z, y, z);
          if (z > x && z > y) d += gram_at(G, M, px, nbf, z, x, z, y);
          if (z > x && y > z) d -= gram_at(G, M, px, nbf, z, x, y, z);
          if (x > z && z > y) d -= gram_at(G, M, px, nbf, x, z, z, y);
          s += G.hr * d;
        }
      }
    }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (threadIdx.x == 0) g1[e] = s;
}

// Ranges of a block's rows at kc roots: about four workgroups per CU in all, 8
// chunks each at least, and at most 256 MB of partial tiles.
struct GramSplit {
  int ntp, nsplit;
  int64_t per;
  size_t part() const { return (size_t)nsplit * ntp * kPT * kPT; }
};
GramSplit gram_split(const RasBlockDev& B, int kc) {
  const int nt = (B.nq + kPT - 1) / kPT, rc = kKK / kc;
  GramSplit g;
  g.ntp = nt * (nt + 1) / 2;
  int64_t n = std::min<int64_t>((1024 + g.ntp - 1) / g.ntp, (B.nrows + 8 * rc - 1) / (8 * rc));
  n = std::max<int64_t>(1, std::min<int64_t>(n, ((int64_t)1 << 25) / ((int64_t)g.ntp * kPT * kPT)));
  g.per = ((B.nrows + n - 1) / n + rc - 1) / rc * rc;
  g.nsplit = (int)((B.nrows + g.per - 1) / g.per);
  return g;
}

template <int KC>
void gram_blocks(Ctx& c, const RasGrad& R, const double* wk, double* part, double* M) {
  const RasPlan& P = c.ras;
  const double* cv = reinterpret_cast<const double*>(c.d_rasc.p);
  for (int bi = 0; bi < (int)P.blk.size(); ++bi) {
    if (R.of[bi] < 0) continue;
    const RasBlockDev& B = P.blk[bi];
    const RasSectorDev& S = P.sec[B.sector];
    // a sector n_alpha > n_beta stands for its spin flip, a product of a
    // symmetric sector for its mirror
    double fac = S.na > S.nb && !P.frac ? 2.0 : 1.0;
    if (S.sym && (B.kind == 1 || B.cu < B.cw || B.tri)) fac *= 2.0;
    const GramSplit g = gram_split(B, KC);
    hipLaunchKernelGGL((k_ras_gram<KC>), dim3((unsigned)g.ntp, (unsigned)g.nsplit), dim3(256), 0, c.stream,
                       c.d_rasview.p, bi, fac, cv, wk, g.per, part);
    PSOCI_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_ras_gram_sum, dim3(nblk((int64_t)g.ntp * kPT * kPT, 256)), dim3(256), 0, c.stream, g.ntp,
                       g.nsplit, part, B.nq, M + R.mat[R.of[bi]].moff);
    PSOCI_HIP(hipGetLastError());
  }
}

}  // namespace

void ras_rdm_grad(Ctx& c, int k, const double* dC, const double* w, double* d_g1, double* d_g2) {
  PSOCI_CHECK(c.have_strings && c.ras_rdm, PSOCI_ERR_STATE, "the string-driven adjoint is not set up");
  const RasPlan& P = c.ras;
  const int nbf = P.nbf;
  const int64_t n1 = (int64_t)nbf * (nbf + 1) / 2, n2 = n1 * (n1 + 1) / 2;
  const RasGrad R = ras_grad(P);
  const std::vector<RasGradMat>& mat = R.mat;
  // the roots in chunks of 16, 8, 4 or 2, their weights padded with zeros
  std::vector<double> hw((size_t)k + 16, 0.0);
  for (int x = 0; x < k; ++x) hw[x] = w ? w[x] : 1.0;
  size_t npart = 0;
  for (int c0 = 0; c0 < k; c0 += c.ras_kc64)
    for (size_t bi = 0; bi < P.blk.size(); ++bi)
      if (R.of[bi] >= 0)
        npart = std::max(npart, gram_split(P.blk[bi], ras_width64(std::min(c.ras_kc64, k - c0))).part());
  SpareUse spare_use(c.spare, 3, 1);
  Scratch arena{c.spare.buf[3]};
  arena.buf.reserve(arena.bytes(npart, 8) + arena.bytes(R.total, 8) + arena.bytes(hw.size(), 8) +
                    arena.bytes(mat.size(), sizeof(RasGradMat)));
  double* part = arena.take<double>(npart);
  double* M = arena.take<double>(R.total);
  double* wk = arena.take<double>(hw.size());
  RasGradMat* dm = arena.take<RasGradMat>(mat.size());
  PSOCI_HIP(hipMemcpyAsync(dm, mat.data(), mat.size() * sizeof(RasGradMat), hipMemcpyHostToDevice, c.stream));
  hipLaunchKernelGGL(k_ras_fill0, dim3(nblk(R.total, 256)), dim3(256), 0, c.stream, R.total, M);
  PSOCI_HIP(hipGetLastError());
  PSOCI_HIP(hipMemcpyAsync(wk, hw.data(), hw.size() * sizeof(double), hipMemcpyHostToDevice, c.stream));
  for (int c0 = 0; c0 < k; c0 += c.ras_kc64) {
    const int kw = std::min(c.ras_kc64, k - c0);
    const int kc = ras_scatter64(c, dC, k, c0, kw);
    const double* wc = wk + c0;
    if (kc == 16) gram_blocks<16>(c, R, wc, part, M);
    else if (kc == 8) gram_blocks<8>(c, R, wc, part, M);
    else if (kc == 4) gram_blocks<4>(c, R, wc, part, M);
    else gram_blocks<2>(c, R, wc, part, M);
  }
  hipLaunchKernelGGL(k_ras_grad2, dim3(nblk(n2, 256)), dim3(256), 0, c.stream, nbf, n2, (int)mat.size(), dm,
                     c.d_raspidx.p, M, d_g2);
  PSOCI_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_ras_grad1, dim3((unsigned)n1), dim3(64), 0, c.stream, nbf, (int)n1, (int)mat.size(), dm,
                     c.d_raspidx.p, M, d_g1);
  PSOCI_HIP(hipGetLastError());
  c.sync();
}

}  // namespace psoci
