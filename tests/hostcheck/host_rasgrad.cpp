// Test harness: the matrices that the string-driven adjoint sums its blocks
// into (ras_grad), against the plan's blocks.  Not part of the product library.
#include "../../psoci_amd/csrc/common.hpp"
#include "../../psoci_amd/csrc/ras.hpp"

using namespace psoci;

// info[0] = blocks, [1] = blocks without pairs, [2] = matrices; 0 on success
extern "C" int hrg_check(int nbf, int nelec, int ksym, int64_t ncfg, const uint8_t* occ, const int32_t* jsym,
                         const double* one, const double* two, int64_t* info) {
  Space sp;
  RasPlan P;
  try {
    build_space(sp, nbf, nelec, ksym, ncfg, occ, jsym);
    ras_plan(P, sp, one, two, true, true);
  } catch (const Error&) {
    return -1;
  }
  if (!P.ok) return 1;
  const RasGrad R = ras_grad(P);
  info[0] = (int64_t)P.blk.size();
  info[1] = 0;
  info[2] = (int64_t)R.mat.size();
  if (R.of.size() != P.blk.size()) return 2;
  std::vector<int> seen(R.mat.size(), -1);
  for (size_t b = 0; b < P.blk.size(); ++b) {
    const RasBlockDev& B = P.blk[b];
    if (B.nq == 0) {
      ++info[1];
      if (R.of[b] != -1) return 3;
      continue;
    }
    const int x = R.of[b];
    if (x < 0 || x >= (int)R.mat.size()) return 4;
    const RasGradMat& G = R.mat[x];
    if (G.nq != B.nq || G.kind != B.kind || G.id != (B.kind ? 1 : 0) * (P.m + 1) + B.budget) return 5;
    if (seen[x] < 0) seen[x] = (int)b;
    const RasBlockDev& F = P.blk[seen[x]];
    if (F.sector != B.sector || F.kind != B.kind || F.budget != B.budget || F.goff != B.goff) return 6;
  }
  // the matrices follow each other and are all used
  int64_t at = 0;
  for (size_t x = 0; x < R.mat.size(); ++x) {
    if (seen[x] < 0 || R.mat[x].nq < 1 || R.mat[x].moff != at) return 7;
    at += (int64_t)R.mat[x].nq * R.mat[x].nq;
  }
  return at == R.total && at > 0 ? 0 : 8;
}

// ras_limit of a plan whose compact and full layouts have these W elements
extern "C" int hrg_limited(int64_t cwunit, int64_t wunit) {
  RasPlan P;
  P.cwunit = P.cdunit = cwunit;
  P.wunit = wunit;
  return ras_limit(P) ? 1 : 0;
}
