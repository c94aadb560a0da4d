// Test harness: the compact layout of the string-driven direct sigma's
// products (RasCmp) evaluated with plain loops on the host CPU.  Not part of
// the product library.
#include <cstring>
#include <vector>

#include "../../psoci_amd/csrc/common.hpp"
#include "../../psoci_amd/csrc/ras.hpp"

using namespace psoci;

// Y[n][k] = H X[n][k] through the compact products; info[0..2] = blocks
// per level, info[3..4] =
// full and compact multiply-adds, info[5] = the list's share of the space.
// general: bit 0 general plans, bit 1 the layouts without dropped pairs.  0
// on success.
extern "C" int hrc_sigma(int nbf, int nelec, int ksym, int64_t ncfg, const uint8_t* occ, const int32_t* jsym,
                         const double* one, const double* two, int k, const double* X, double* Y, double* info,
                         int general) {
  Space sp;
  RasPlan P;
  try {
    build_space(sp, nbf, nelec, ksym, ncfg, occ, jsym);
    ras_plan(P, sp, one, two, (general & 1) != 0, true);
    if (P.ok && (general & 2)) ras_compact(P, true);
  } catch (const Error&) {
    return -1;
  }
  if (!P.ok) return 1;
  RasView v = ras_host_view(P);
  v.cmp = P.cmp.data();
  v.wunit = P.cwunit;
  const double r = 0x1.6a09e667f3bcdp-1;
  std::vector<double> c((size_t)P.ndet * k, 0.0);
  for (int64_t s = 0; s < v.nsef; ++s) {
    const RasSef& e = v.sef[s];
    for (int t = 0; t < e.n; ++t) {
      const RasSectorDev& S = v.sec[e.sec[t]];
      const int ca = ras_cls_of(v, S.na, e.a[t]), cb = ras_cls_of(v, S.nb, e.b[t]);
      const int64_t d = ras_det(v, e.sec[t], ca, e.a[t] - v.lev[S.na].cls_off[ca], cb, e.b[t] - v.lev[S.nb].cls_off[cb]);
      for (int j = 0; j < k; ++j)
        c[d * k + j] = ((e.flag[t] & 2) ? 1.0 : r) * ((e.flag[t] & 1) ? -1.0 : 1.0) * X[s * k + j];
    }
  }
  std::vector<double> W((size_t)P.cwunit * k, 1e300);
  info[0] = info[1] = info[2] = 0.0;
  info[3] = P.gemm_flops_per_col;
  info[4] = P.cflops_per_col;
  info[5] = P.fill;
  for (int bi = 0; bi < v.nblk; ++bi) {
    const RasBlockDev& B = v.blk[bi];
    const RasCmp& C = P.cmp[bi];
    info[C.level] += 1.0;
    if (C.nqp % 16 || C.nq > C.nqp || C.nq > B.nq) return 6;
    // groups cover the rows once, in order, and a row's variant is its group's
    int64_t next = 0;
    int bad = 0;
    std::vector<int64_t> var(C.nrows, -1);
    ras_cmp_groups(C, [&](int64_t g, int64_t r0, int64_t rows) {
      if (r0 != next || g < 0 || g >= C.nvar) bad = 1;
      for (int64_t x = r0; x < r0 + rows && x < C.nrows; ++x) var[x] = g;
      next = r0 + rows;
    });
    if (bad || next != C.nrows) return 7;
    const int16_t* pidx = v.pidx + (size_t)((C.kind ? 1 : 0) * (v.m + 1) + C.budget) * nbf * nbf;
    for (int64_t row = 0; row < C.nrows; ++row) {
      int64_t o, i;
      ras_cmp_unrow(C, row, o, i);
      if (ras_cmp_row(C, o, i) != row) return 8;
      const int64_t oi = o / C.nEo, ii = i / C.nEi;
      if (ras_cmp_var(C, oi, ii) != var[row]) return 9;
      uint64_t op, ir;
      ras_cmp_drop(v, C, oi, ii, op, ir);
      int64_t r0, rows;
      ras_cmp_group(C, oi, ii, r0, rows);
      if (row < r0 || row >= r0 + rows) return 11;
      std::vector<double> D((size_t)C.nq * k, 0.0);
      std::vector<int> full(C.nq, -1);
      int n = 0;
      const int64_t u = (C.swap ? i + C.i0 : o + C.o0), w = (C.swap ? o + C.o0 : i + C.i0);
      ras_cmp_pairs(v, C, op, ir, [&](int j, int p, int q) {
        if (j != n++ || j >= C.nq || ras_cmp_pair(v, C, op, ir, p, q) != j) {
          bad = 1;
          return;
        }
        full[j] = pidx[p * nbf + q];
        int neg = 0;
        const int64_t d = ras_d_det(v, C.kind, C.sector, B.lu, B.lw, u, w, p, q, neg);
        if (d >= P.ndet || full[j] < 0) bad = 1;
        else if (d >= 0)
          for (int t = 0; t < k; ++t) D[(size_t)j * k + t] = neg ? -c[d * k + t] : c[d * k + t];
      });
      if (bad || n != C.nq) return 10;
      const double* G = P.G.data() + B.goff;
      for (int a = 0; a < C.nq; ++a)
        for (int t = 0; t < k; ++t) {
          double acc = 0.0;
          for (int j = 0; j < C.nq; ++j) acc += G[(int64_t)full[a] * B.nqp + full[j]] * D[(size_t)j * k + t];
          W[ras_cmp_w(C, r0, rows, row, a) * k + t] = acc;
        }
    }
  }
  const double sc[3] = {r, 1.0 / r, 1.0};
  for (int64_t s = 0; s < v.nsef; ++s) {
    int bad = 0;
    std::vector<double> sig(k, 0.0);
    const int code = ras_sef_terms(v, v.sef[s], &bad, [&](int64_t off, int neg) {
      for (int q = 0; q < k; ++q) sig[q] += neg ? -W[off * k + q] : W[off * k + q];
    });
    if (bad) return 5;
    for (int q = 0; q < k; ++q) Y[s * k + q] = sc[code] * sig[q];
  }
  return 0;
}
