// Hamiltonian construction on the GPU: pair screening, configuration-pair
// setup, SEF element generation and deterministic compaction into CSR.
//
// Replaces constructGlobalHamiltonianAltOrbMapDirectChunkJmap with
// packSefsef (PsociGAhamiltonian.C:2530-2857, 4077-4136).  The reference's
// row for SEF i of configuration I lists, for J <= I ascending (one J chunk),
// the elements of block (I, J) row i with |h| >= 1e-8 (and the diagonal),
// columns ascending.  Here the blocks' kept elements are a bit string and a
// value array in block order; a wavefront per row counts the bits of the
// row's segments, a prefix sum over the rows gives the CSR offsets, and the
// same walk writes the elements -- their places follow from the bits alone,
// so the result is bit-for-bit reproducible.
//
// The context keeps the symmetric full matrix: row r holds its lower part
// (the reference's row, diagonal last) followed by the transposed elements of
// blocks (I, J) with I > J, ascending.
#include <chrono>
#include <hipcub/hipcub.hpp>

#include "ctx.hpp"

namespace psoci {

namespace {

constexpr int kWave = 64;
constexpr double kThresh = 1.0e-8;  // MIN_DOUBLE_VALUE (PsociHamiltonian.hpp:37)

// the configuration's determinant patterns come from its class's family
// (12 offsets per family)
__device__ __forceinline__ ConfView conf_view(int64_t c, const uint64_t* dm, const uint64_t* sm, const int8_t* nopen,
                                              const uint8_t* cph, const uint16_t* pat, const int32_t* patoff,
                                              const uint8_t* cls) {
  ConfView v;
  v.d = dm[c];
  v.s = sm[c];
  v.nopen = nopen[c];
  v.ph = cph[c];
  v.pat = pat + patoff[12 * cls[c] + v.nopen];
  return v;
}

// One wavefront per configuration I: ballot over candidate J, ascending.  The
// connected J <= I (the reference's J list, compareLocalJSubsetOrbMap,
// PsociGADeterminants.C:2501-2546) and those above I, in one walk: a list of
// J <= I alone takes the last wavefronts as long and leaves the first idle.
// FILL = false counts them (cnt[I], cnt[ncfg + I]); FILL = true lists them at
// their offsets in the prefix sum of those counts, with the row configuration
// and the block size of the lower pairs.
template <bool FILL>
__global__ void k_screen(int64_t ncfg, const uint64_t* __restrict__ dm, const uint64_t* __restrict__ sm,
                         const int8_t* __restrict__ nopen, const int32_t* __restrict__ nsef,
                         int64_t* __restrict__ cnt, const int64_t* __restrict__ off, int32_t* __restrict__ list,
                         int32_t* __restrict__ rowcfg, int64_t* __restrict__ blk_size) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t I = (int64_t)blockIdx.x * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (I >= ncfg) return;  // uniform per wavefront
  const uint64_t dI = dm[I], sI = sm[I];
  const int nI = nopen[I];
  const int64_t eI = nsef[I];
  int64_t lo = FILL ? off[I] : 0, up = FILL ? off[ncfg + I] : 0;
  for (int64_t J0 = 0; J0 < ncfg; J0 += kWave) {
    const int64_t J = J0 + lane;
    bool ok = false;
    if (J < ncfg) {
      int dn = nI - nopen[J];
      if (dn <= 4 && dn >= -4) ok = moved(dI, sI, dm[J], sm[J]) <= 2;
    }
    const uint64_t ml = __ballot(ok && J <= I), mu = __ballot(ok && J > I);
    if (FILL && ok) {
      const uint64_t below = (1ull << lane) - 1ull;
      if (J <= I) {
        const int64_t p = lo + popc(ml & below);
        list[p] = (int32_t)J;
        rowcfg[p] = (int32_t)I;
        blk_size[p] = eI * nsef[J];
      } else {
        list[up + popc(mu & below)] = (int32_t)J;
      }
    }
    lo += popc(ml);
    up += popc(mu);
  }
  if (!FILL && lane == 0) {
    cnt[I] = lo;
    cnt[ncfg + I] = up;
  }
}

__global__ void k_pair_setup(int64_t npairs, const int32_t* __restrict__ rowcfg, const int32_t* __restrict__ colcfg,
                             const uint64_t* __restrict__ dm, const uint64_t* __restrict__ sm,
                             const int8_t* __restrict__ nopen, const int32_t* __restrict__ jsym, int nbf,
                             const double* __restrict__ one, const double* __restrict__ two,
                             PairInfo* __restrict__ pairs) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npairs) return;
  int I = rowcfg[p], J = colcfg[p];
  PairInfo P;
  pair_setup(P, I, J, dm[I], sm[I], nopen[I], dm[J], sm[J], nopen[J], nbf, one, two, jsym[I], jsym[J]);
  pairs[p] = P;
}

// Per SEF: its configuration and the alpha set of its first determinant
// (determinant 2k of an even-electron configuration, whose partner 2k + 1 has
// every open shell's spin flipped; determinant k of an odd one).
__global__ void k_sef_masks(int64_t ncfg, const uint64_t* __restrict__ dm, const uint64_t* __restrict__ sm,
                            const int8_t* __restrict__ nopen, const uint16_t* __restrict__ pat,
                            const int32_t* __restrict__ patoff, const uint8_t* __restrict__ cls,
                            const int32_t* __restrict__ nsef, const int64_t* __restrict__ sefoff, int frac,
                            uint64_t* __restrict__ amask, int32_t* __restrict__ cfg) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t I = (int64_t)blockIdx.x * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (I >= ncfg) return;
  const uint64_t d = dm[I], s = sm[I];
  const int step = (frac || nopen[I] == 0) ? 1 : 2;
  const uint16_t* pt = pat + patoff[12 * cls[I] + nopen[I]];
  for (int i = lane; i < nsef[I]; i += kWave) {
    amask[sefoff[I] + i] = d | deposit(pt[step * i], s);
    cfg[sefoff[I] + i] = (int32_t)I;
  }
}

// Elements per wavefront of k_block_elems.  Eight 64-element steps fill the
// queue of connected elements far enough that its last, partly filled
// evaluation costs little (about one element in ten is connected).
constexpr int kBatch = 512;

// first[b]: the pair that holds element b * kBatch
__global__ void k_batch_first(int64_t npairs, const int64_t* __restrict__ blk_off, int64_t* __restrict__ first) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npairs) return;
  const int64_t e1 = blk_off[p + 1];
  for (int64_t b = (blk_off[p] + kBatch - 1) / kBatch; b * kBatch < e1; ++b) first[b] = p;
}

// orders a wavefront's own LDS traffic
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Two determinants (alpha sets a and b; sx = the XOR of their configurations'
// open shells) within two replacements and of one spin projection: the beta
// set is the alpha set XOR the open shells.
__device__ __forceinline__ bool connected(uint64_t a, uint64_t b, uint64_t sx) {
  const uint64_t x = a ^ b;
  return popc(x) + popc(x ^ sx) <= 4 && popc(a) == popc(b);
}

// The pairs of a wavefront's steps of 64 elements: the lanes mark the block
// boundaries among the step's elements (mark: a wavefront's 64 words of LDS),
// a ballot and a count give each lane its pair.
struct PairWalk {
  int64_t p0, next;  // the step's first pair and its end
  __device__ __forceinline__ PairWalk(int64_t p, const int64_t* __restrict__ blk_off) : p0(p), next(blk_off[p + 1]) {}
  __device__ __forceinline__ int64_t step(int64_t es, int lane, uint32_t* mark, int64_t npairs,
                                          const int64_t* __restrict__ blk_off) {
    if (next - es > kWave) return p0;
    // boundaries past p0's first element (all at 1 or later)
    mark[lane] = 0;
    lds_order();
    const int64_t pb = p0 + 1 + lane;
    const int64_t left = pb <= npairs ? blk_off[pb] - es : kWave + 1;
    if (left < kWave) mark[left] = 1;
    lds_order();
    const int64_t p = p0 + popc(__ballot(mark[lane] != 0) & ((2ull << lane) - 1ull));
    p0 += popc(__ballot(left <= kWave));
    if (p0 < npairs) next = blk_off[p0 + 1];
    return p;
  }
};

// Elements of the blocks, in block order: element (i, j) of pair p is number
// blk_off[p] + i * nsef_J + j.  Kept ones (|h| >= 1e-8, and the diagonal; of
// a diagonal block its lower triangle) get their bit; their values stand
// together at the start of each batch of kBatch elements (staging), and
// rank[w] counts those of the batch before word w of the bits.  Values left at
// their own elements cost the rows' gather a memory line each.
//
// One wavefront per 512 elements.  Bound by vector instructions: a
// determinant pair's evaluation is some 150 and about one element in ten is
// connected at all, so each 64-element step only tests its elements (the XOR
// of two 64-bit masks and its counts) and appends the connected ones to a
// queue in LDS; the queue is then evaluated 64 at a time, every lane with
// work.  Of an even-electron element's four determinant pairs two are
// evaluated: flipping every open spin on both sides leaves a determinant
// pair's element as it is, bit for bit (spin-orbit pairs take all four).
// Measured on full CI of 10 orbitals and 8 electrons (31,650 SEFs, 78 M
// elements): 0.44 ms; a thread per element, with its own search for its pair
// and four evaluations, took 2.24 ms.
template <bool FRAC>
__global__ __launch_bounds__(256) void k_block_elems(
    int64_t total, int64_t npairs, const int64_t* __restrict__ blk_off, const int64_t* __restrict__ first,
    const PairInfo* __restrict__ pairs, const uint64_t* __restrict__ dm, const uint64_t* __restrict__ sm,
    const int8_t* __restrict__ nopen, const uint8_t* __restrict__ cph, const double* __restrict__ cmult,
    const int32_t* __restrict__ nsef, const int64_t* __restrict__ sefoff, const uint64_t* __restrict__ amask,
    const double* __restrict__ two, double* __restrict__ staging, uint64_t* __restrict__ bits,
    uint16_t* __restrict__ rank) {
  __shared__ uint32_t sh_mark[4][kWave];
  __shared__ uint32_t sh_queue[4][kBatch];
  __shared__ uint32_t sh_bits[4][kBatch / 32];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t batch = (int64_t)blockIdx.x * (blockDim.x / kWave) + wv;
  const int64_t e0 = batch * kBatch;
  if (e0 >= total) return;  // uniform per wavefront; no workgroup barrier below
  uint32_t* mark = sh_mark[wv];
  uint32_t* queue = sh_queue[wv];
  uint32_t* wb = sh_bits[wv];
  const int64_t pf = first[batch];
  PairWalk walk(pf, blk_off);
  int nq = 0;
  if (lane < kBatch / 32) wb[lane] = 0;
  // the lane's pair: kept while its elements stay in it (a block of more than
  // 64 elements gives a lane several)
  int64_t pc = -1, off = 0;
  int sh = 0, kind = 0;
  bool diag = false;
  const uint64_t *ai = nullptr, *aj = nullptr;
  uint64_t sj = 0, sx = 0;
  for (int c = 0; c < kBatch / kWave; ++c) {
    const int64_t es = e0 + c * kWave;
    if (es >= total) break;
    const int64_t p = walk.step(es, lane, mark, npairs, blk_off);
    const int64_t e = es + lane;
    bool ok = false;
    if (e < total) {
      if (p != pc) {
        pc = p;
        off = blk_off[p];
        const int I = pairs[p].I, J = pairs[p].J;
        kind = pairs[p].kind;
        diag = I == J;
        sh = popc((uint64_t)(nsef[J] - 1));  // a configuration's SEFs are a power of two
        ai = amask + sefoff[I];
        aj = amask + sefoff[J];
        sj = sm[J];
        sx = sm[I] ^ sj;
      }
      const unsigned loc = (unsigned)(e - off), i = loc >> sh, j = loc - (i << sh);
      if (kind != 0 && (!diag || j <= i)) {
        const uint64_t a = ai[i], b = aj[j];
        ok = kind == 4 || connected(a, b, sx) || (!FRAC && connected(a, b ^ sj, sx));
      }
    }
    const uint64_t mo = __ballot(ok);
    if (ok) queue[nq + popc(mo & ((1ull << lane) - 1ull))] = (uint32_t)(c * kWave + lane) | (uint32_t)(p - pf) << 16;
    nq += popc(mo);
  }
  lds_order();
  int kept = 0;
  for (int k0 = 0; k0 < nq; k0 += kWave) {
    double v = 0.0;
    unsigned rel = 0;
    bool keep = false;
    if (k0 + lane < nq) {
      const uint32_t ent = queue[k0 + lane];
      rel = ent & 0xffffu;
      const int64_t p = pf + (ent >> 16);
      const PairInfo P = pairs[p];
      const unsigned loc = (unsigned)(e0 + rel - blk_off[p]);
      const int sh = popc((uint64_t)(nsef[P.J] - 1));
      const unsigned i = loc >> sh, j = loc - (i << sh);
      ConfView A{dm[P.I], sm[P.I], nopen[P.I], cph[P.I], nullptr}, B{dm[P.J], sm[P.J], nopen[P.J], cph[P.J], nullptr};
      const uint64_t a0 = amask[sefoff[P.I] + i] & A.s, b0 = amask[sefoff[P.J] + j] & B.s;
      if (FRAC)
        v = detval_ao(P, A, B, a0, b0, two);
      else if (P.kind == 4)
        v = sef_elem_ao(P, A, B, a0, A.s & ~a0, b0, B.s & ~b0, cmult[P.I], cmult[P.J], two);
      else
        v = sef_elem_flip(P, A, B, a0, b0, cmult[P.I], cmult[P.J], two);
      keep = fabs(v) >= kThresh || (P.I == P.J && i == j);
    }
    // the queue is in element order, and so are the values
    const uint64_t mk = __ballot(keep);
    if (keep) {
      staging[e0 + kept + popc(mk & ((1ull << lane) - 1ull))] = v;
      atomicOr(&wb[rel >> 5], 1u << (rel & 31));
    }
    kept += popc(mk);
  }
  lds_order();
  if (lane < kBatch / 64) {
    const int64_t w = e0 / 64 + lane;
    int before = 0;
    for (int q = 0; q < 2 * lane; ++q) before += __builtin_popcount(wb[q]);
    if (w * 64 < total) {
      bits[w] = (uint64_t)wb[2 * lane + 1] << 32 | wb[2 * lane];
      rank[w] = (uint16_t)before;
    }
  }
}

// The same bits with each block transposed: element (i, j) of pair p is bit
// blk_off[p] + j * nsef_I + i.  One wavefront per 512 bits, a lane fetches
// the source bit of one of a step's 64; bound by the latency of the
// walk over the blocks (0.15 ms for 78 M bits; set one by one with atomics
// where the elements are evaluated they took 0.21 ms).
__global__ __launch_bounds__(256) void k_transpose_bits(int64_t total, int64_t npairs,
                                                        const int64_t* __restrict__ blk_off,
                                                        const int64_t* __restrict__ first,
                                                        const PairInfo* __restrict__ pairs,
                                                        const int32_t* __restrict__ nsef,
                                                        const uint64_t* __restrict__ bits,
                                                        uint64_t* __restrict__ tbits) {
  __shared__ uint32_t sh_mark[4][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t batch = (int64_t)blockIdx.x * (blockDim.x / kWave) + wv;
  const int64_t e0 = batch * kBatch;
  if (e0 >= total) return;  // uniform per wavefront; no workgroup barrier below
  PairWalk walk(first[batch], blk_off);
  int64_t pc = -1, off = 0;
  int shi = 0, shj = 0;
  // all source words are fetched before the first is used
  uint64_t word[kBatch / kWave];
  int at[kBatch / kWave];
#pragma unroll
  for (int c = 0; c < kBatch / kWave; ++c) {
    const int64_t es = e0 + c * kWave, e = es + lane;
    word[c] = 0;
    at[c] = 0;
    if (es < total) {
      const int64_t p = walk.step(es, lane, sh_mark[wv], npairs, blk_off);
      if (e < total) {
        if (p != pc) {
          pc = p;
          off = blk_off[p];
          shi = popc((uint64_t)(nsef[pairs[p].I] - 1));
          shj = popc((uint64_t)(nsef[pairs[p].J] - 1));
        }
        const unsigned loc = (unsigned)(e - off), j = loc >> shi, i = loc - (j << shi);
        const int64_t src = off + ((i << shj) | j);
        at[c] = (int)(src & 63);
        word[c] = bits[src >> 6];
      }
    }
  }
  uint64_t out = 0;  // lane c's word of the batch
#pragma unroll
  for (int c = 0; c < kBatch / kWave; ++c) {
    const uint64_t m = __ballot(word[c] >> at[c] & 1ull);
    if (lane == c) out = m;
  }
  if (lane < kBatch / 64 && e0 + lane * 64 < total) tbits[e0 / 64 + lane] = out;
}

// One segment of a configuration's rows: the block that holds it.  Row j's
// elements are, in segment order, row j of the block of a lower pair, or
// column j of the block of an upper pair.
struct Seg {
  int64_t off;  // first element of the block
  int32_t col;  // first SEF of the other configuration
  int32_t len;  // its SEFs; 0 where the block is skipped
};
static_assert(sizeof(Seg) == 16, "Seg layout");

__device__ __forceinline__ int64_t find_pair(const int32_t* __restrict__ colcfg, int64_t lo, int64_t hi, int32_t J) {
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    if (colcfg[mid] < J) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// The segments of configuration J: its lower pairs (the diagonal block last),
// the diagonal block again for the transposed elements of its lower triangle,
// then the upper pairs.  The lists are the configurations' lower pairs, then
// their upper pairs (off: the offsets of both).
struct RowSegs {
  int64_t l0, u0;  // the lists of the lower and the upper pairs
  int64_t s0;      // the segments
  int nl, w;       // lower pairs; segments
};

__device__ __forceinline__ RowSegs row_segs(int64_t J, int64_t ncfg, const int64_t* __restrict__ off) {
  RowSegs m;
  m.l0 = off[J];
  m.u0 = off[ncfg + J];
  m.s0 = m.l0 + (m.u0 - off[ncfg]) + J;
  m.nl = (int)(off[J + 1] - m.l0);
  m.w = m.nl + 1 + (int)(off[ncfg + J + 1] - m.u0);
  return m;
}

// Each upper pair is looked up once here and not once per row.
__global__ __launch_bounds__(256) void k_segs(int64_t ncfg, const int64_t* __restrict__ off,
                                              const int32_t* __restrict__ list, const PairInfo* __restrict__ pairs,
                                              const int64_t* __restrict__ blk_off, const int32_t* __restrict__ nsef,
                                              const int64_t* __restrict__ sefoff, Seg* __restrict__ segs) {
  const int64_t J = blockIdx.x;
  const RowSegs m = row_segs(J, ncfg, off);
  for (int t = threadIdx.x; t < m.w; t += blockDim.x) {
    int64_t p;
    int32_t K;
    bool found = true;
    if (t <= m.nl) {
      p = m.l0 + (t < m.nl ? t : m.nl - 1);
      K = list[p];
    } else {
      K = list[m.u0 + (t - m.nl - 1)];
      p = find_pair(list, off[K], off[K + 1], (int32_t)J);
      // the predicate is symmetric, so (K, J) is in K's lower list; guard anyway
      found = p < off[K + 1] && list[p] == (int32_t)J;
    }
    Seg s;
    s.off = found ? blk_off[p] : 0;
    s.col = (int32_t)sefoff[K];
    s.len = found && pairs[p].kind != 0 ? nsef[K] : 0;
    segs[m.s0 + t] = s;
  }
}

// 64 bits from bit position pos (two padding words follow the last)
__device__ __forceinline__ uint64_t bits_at(const uint64_t* __restrict__ bits, int64_t pos) {
  const int64_t w = pos >> 6;
  const int s = (int)(pos & 63);
  const uint64_t lo = bits[w], hi = bits[w + 1];
  return s ? lo >> s | hi << (64 - s) : lo;
}

// The rows of the full matrix, one wavefront per row, a lane per segment and
// turn of 64 segments: FILL = false counts a row's kept elements, FILL = true
// writes them at the row's offset, a prefix sum over the turn's lanes giving
// each segment's place.  A segment is a run of bits: of the blocks' bits for
// a lower pair, of the transposed ones for an upper pair (walking block
// columns in the one array took several dependent loads a segment and bound
// the walk by their latency: 0.29 ms for the counts, 0.07 ms so).  The values'
// gather is bound by the lines it misses in L2: 0.34 ms for 11 M elements at
// 5 to 6 TB/s.  A thread per (row, pair) segment, each searching for its row
// and pair, took 1.69 ms for the counts and 1.91 ms for the elements, and a
// prefix sum over 18 M segments.
template <bool FILL>
__global__ __launch_bounds__(256) void k_rows(
    int64_t n, int64_t ncfg, const int32_t* __restrict__ cfg, const int64_t* __restrict__ off,
    const int32_t* __restrict__ nsef, const int64_t* __restrict__ sefoff, const Seg* __restrict__ segs,
    const uint64_t* __restrict__ bits, const uint64_t* __restrict__ tbits, const uint16_t* __restrict__ rank,
    const double* __restrict__ staging, int64_t* __restrict__ cnt, const int64_t* __restrict__ rowptr,
    int32_t* __restrict__ col, double* __restrict__ val, float* __restrict__ val32, int32_t* __restrict__ lowcnt,
    double* __restrict__ diag) {
  const int lane = threadIdx.x & (kWave - 1);
  // 64 consecutive rows to an XCD (workgroups go to the eight in turn): the
  // rows of a configuration read the same blocks' bits and values
  const int64_t q8 = blockIdx.x >> 3, b = ((q8 >> 4) * 8 + (blockIdx.x & 7)) * 16 + (q8 & 15);
  const int64_t r = b * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (r >= n) return;  // uniform per wavefront
  const int64_t J = cfg[r];
  const RowSegs m = row_segs(J, ncfg, off);
  const int nl = m.nl, w = m.w;
  const int nj = nsef[J], j = (int)(r - sefoff[J]);
  const Seg* sg = segs + m.s0;
  // the value of the kept element number pos
  auto value = [&](int64_t pos) {
    const int64_t bw = pos >> 6;
    return staging[bw / (kBatch / 64) * kBatch + rank[bw] + popc(bits[bw] & ((1ull << (pos & 63)) - 1ull))];
  };
  // a row's next elements (number and column) wait in LDS, so that the values
  // are gathered and stored by whole wavefronts
  constexpr int kList = 256;
  __shared__ int64_t sh_pos[FILL ? 4 : 1][FILL ? kList : 1];
  __shared__ int32_t sh_col[FILL ? 4 : 1][FILL ? kList : 1];
  int64_t* lpos = sh_pos[FILL ? threadIdx.x / kWave : 0];
  int32_t* lcol = sh_col[FILL ? threadIdx.x / kWave : 0];
  const int64_t row0 = FILL ? rowptr[r] : 0;
  int64_t at = row0;  // where the list's first element goes
  int have = 0;       // its length
  auto flush = [&] {
    lds_order();
    for (int k = lane; k < have; k += kWave) {
      const double v = value(lpos[k]);
      col[at + k] = lcol[k];
      val[at + k] = v;
      val32[at + k] = (float)v;
    }
    lds_order();
    at += have;
    have = 0;
  };
  int total = 0;
  for (int t0 = 0; t0 < w; t0 += kWave) {
    const int t = t0 + lane;
    Seg s{0, 0, 0};
    if (t < w) s = sg[t];
    const bool low = t < nl;
    const int64_t start = s.off + (int64_t)j * s.len;
    const int q0 = t == nl ? j + 1 : 0;  // the transposed lower triangle
    auto word = [&](int q) {
      const uint64_t b = bits_at(low ? bits : tbits, start + q);
      return s.len - q < 64 ? b & ((1ull << (s.len - q)) - 1ull) : b;
    };
    const uint64_t b0 = q0 < s.len ? word(q0) : 0;
    int c = popc(b0);
    for (int q = q0 + 64; q < s.len; q += 64) c += popc(word(q));
    if (FILL) {
      int pre = c;  // inclusive prefix over the lanes
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const int up = __shfl_up(pre, o);
        if (lane >= o) pre += up;
      }
      const int turn = __shfl(pre, kWave - 1);
      // the diagonal element ends the lower part of the row
      if (t == nl - 1) {
        lowcnt[r] = (int32_t)(at + have + pre - row0);
        diag[r] = value(start + j);
      }
      for (int done = 0; done < turn;) {
        const int put = turn - done < kList - have ? turn - done : kList - have;
        int idx = pre - c - done;  // place of the lane's next element from done on
        for (int q = q0; q < s.len && idx < put; q += 64) {
          uint64_t x = q == q0 ? b0 : word(q);
          while (x) {
            const int qq = q + ctz(x);
            x &= x - 1;
            if (idx >= 0 && idx < put) {
              lpos[have + idx] = low ? start + qq : s.off + (int64_t)qq * nj + j;
              lcol[have + idx] = s.col + qq;
            }
            ++idx;
          }
        }
        have += put;
        done += put;
        if (have == kList) flush();
      }
    } else {
      total += c;
    }
  }
  if (FILL) {
    flush();
  } else {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) total += __shfl_xor(total, o);
    if (lane == 0) cnt[r] = total;
  }
}

__global__ void k_to_f32(int64_t n, const double* __restrict__ a, float* __restrict__ b) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) b[t] = (float)a[t];
}

// diagonal only: computeOnlyDiagElements (PsociGAhamiltonian.C:13171-13250)
__global__ void k_diag_only(int64_t ncfg, const uint64_t* __restrict__ dm, const uint64_t* __restrict__ sm,
                            const int8_t* __restrict__ nopen, const uint8_t* __restrict__ cph,
                            const uint16_t* __restrict__ pat, const int32_t* __restrict__ patoff,
                            const uint8_t* __restrict__ cls, const double* __restrict__ cmult,
                            const int32_t* __restrict__ nsef, const int64_t* __restrict__ sefoff, int nbf, int frac,
                            const double* __restrict__ one, const double* __restrict__ two,
                            double* __restrict__ diag) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t I = (int64_t)blockIdx.x * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (I >= ncfg) return;
  PairInfo P;
  if (lane == 0) pair_setup(P, (int)I, (int)I, dm[I], sm[I], nopen[I], dm[I], sm[I], nopen[I], nbf, one, two);
  P.v0 = __shfl(P.v0, 0, kWave);
  P.kind = 1;
  P.I = P.J = (int)I;
  ConfView A = conf_view(I, dm, sm, nopen, cph, pat, patoff, cls);
  const double mult = cmult[I];
  for (int i = lane; i < nsef[I]; i += kWave) diag[sefoff[I] + i] = sef_elem(P, A, A, i, i, mult, mult, two, frac != 0);
}

__global__ void k_single_block(PairInfo* __restrict__ Pout, int I, int J, const uint64_t* __restrict__ dm,
                               const uint64_t* __restrict__ sm, const int8_t* __restrict__ nopen,
                               const uint8_t* __restrict__ cph, const uint16_t* __restrict__ pat,
                               const int32_t* __restrict__ patoff, const uint8_t* __restrict__ cls,
                               const double* __restrict__ cmult, const int32_t* __restrict__ jsym,
                               const int32_t* __restrict__ nsef, int nbf, int frac, const double* __restrict__ one,
                               const double* __restrict__ two, double* __restrict__ out) {
  __shared__ PairInfo P;
  if (threadIdx.x == 0) {
    pair_setup(P, I, J, dm[I], sm[I], nopen[I], dm[J], sm[J], nopen[J], nbf, one, two, jsym[I], jsym[J]);
    *Pout = P;
  }
  __syncthreads();
  ConfView A = conf_view(I, dm, sm, nopen, cph, pat, patoff, cls);
  ConfView B = conf_view(J, dm, sm, nopen, cph, pat, patoff, cls);
  int ni = nsef[I], nj = nsef[J];
  for (int e = threadIdx.x; e < ni * nj; e += blockDim.x) {
    int i = e / nj, j = e - i * nj;
    out[e] = (P.kind != 0) ? sef_elem(P, A, B, i, j, cmult[I], cmult[J], two, frac != 0) : 0.0;
  }
}

__global__ void k_extract_lower(int64_t n, const int64_t* __restrict__ rowptr, const int32_t* __restrict__ lowcnt,
                                const int64_t* __restrict__ lowptr, const int32_t* __restrict__ col,
                                const double* __restrict__ val, int32_t* __restrict__ lcol, double* __restrict__ lval) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t r = (int64_t)blockIdx.x * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (r >= n) return;
  int64_t a = rowptr[r], b = lowptr[r];
  for (int q = lane; q < lowcnt[r]; q += kWave) {
    lcol[b + q] = col[a + q];
    lval[b + q] = val[a + q];
  }
}

inline unsigned blocks_for(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

void exclusive_scan_i64(const int64_t* in, int64_t* out, int64_t n, hipStream_t s, void*& tmp, size_t& tmp_bytes) {
  if (n <= 0) return;
  size_t need = 0;
  PSOCI_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, need, in, out, (int)0 + n, s));
  if (need > tmp_bytes) {
    if (tmp) PSOCI_HIP(hipFree(tmp));
    tmp = nullptr;
    PSOCI_HIP(device_malloc(&tmp, need));
    tmp_bytes = need;
  }
  PSOCI_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tmp_bytes, in, out, n, s));
}

void upload_space(Ctx& c) {
  const Space& sp = c.sp;
  c.d_dm.upload(sp.dm, c.stream);
  c.d_sm.upload(sp.sm, c.stream);
  c.d_nopen.upload(sp.nopen, c.stream);
  c.d_nsef.upload(sp.nsef, c.stream);
  c.d_sefoff.upload(sp.sef_off, c.stream);
  c.d_cph.upload(sp.cphase, c.stream);
  c.d_pat.upload(sp.pat, c.stream);
  std::vector<int32_t> po(sp.pat_off, sp.pat_off + 24);
  c.d_patoff.upload(po, c.stream);
  c.d_didx.upload(sp.didx, c.stream);
  c.d_cls.upload(sp.cls, c.stream);
  c.d_cmult.upload(sp.cmult, c.stream);
  c.d_jsym.upload(sp.jsym, c.stream);
  c.sync();
}

void build_h(Ctx& c) {
  const Space& sp = c.sp;
  const int64_t ncfg = sp.ncfg, n = sp.nsef_total;
  const auto t0 = std::chrono::steady_clock::now();
  SpareUse spare_use(c.spare, 0, 2);
  // connected pairs: lower (J <= I per I), then upper (J > I)
  DevBuf<int64_t> cnt, off;
  cnt.alloc(std::max(2 * ncfg, n) + 1);
  off.alloc(2 * ncfg + 1);
  const unsigned per_cfg = blocks_for(ncfg, 4);  // a wavefront per configuration
  PSOCI_HIP(hipMemsetAsync(cnt.p + 2 * ncfg, 0, sizeof(int64_t), c.stream));
  hipLaunchKernelGGL(k_screen<false>, dim3(per_cfg), dim3(256), 0, c.stream, ncfg, c.d_dm.p, c.d_sm.p, c.d_nopen.p,
                     c.d_nsef.p, cnt.p, nullptr, nullptr, nullptr, nullptr);
  PSOCI_HIP(hipGetLastError());
  c.scan(cnt.p, off.p, 2 * ncfg + 1);
  int64_t np = 0, nboth = 0;
  PSOCI_HIP(hipMemcpyAsync(&np, off.p + ncfg, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
  PSOCI_HIP(hipMemcpyAsync(&nboth, off.p + 2 * ncfg, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
  c.sync();
  Scratch sa{c.spare.buf[0]};
  sa.buf.reserve(sa.bytes(nboth, 4) + sa.bytes(np, 4) + sa.bytes(np, sizeof(PairInfo)) + 2 * sa.bytes(np + 1, 8) +
               sa.bytes(nboth + ncfg, sizeof(Seg)));
  int32_t* list = sa.take<int32_t>(nboth);
  int32_t* rowcfg = sa.take<int32_t>(np);
  PairInfo* info = sa.take<PairInfo>(np);
  int64_t* bsz = sa.take<int64_t>(np + 1);
  int64_t* boff = sa.take<int64_t>(np + 1);
  Seg* segs = sa.take<Seg>(nboth + ncfg);
  PSOCI_HIP(hipMemsetAsync(bsz + np, 0, sizeof(int64_t), c.stream));
  hipLaunchKernelGGL(k_screen<true>, dim3(per_cfg), dim3(256), 0, c.stream, ncfg, c.d_dm.p, c.d_sm.p, c.d_nopen.p,
                     c.d_nsef.p, nullptr, off.p, list, rowcfg, bsz);
  PSOCI_HIP(hipGetLastError());
  c.scan(bsz, boff, np + 1);
  int64_t nstage = 0;
  PSOCI_HIP(hipMemcpyAsync(&nstage, boff + np, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
  hipLaunchKernelGGL(k_pair_setup, dim3(blocks_for(np, 256)), dim3(256), 0, c.stream, np, rowcfg, list, c.d_dm.p,
                     c.d_sm.p, c.d_nopen.p, c.d_jsym.p, sp.nbf, c.d_one.p, c.d_two.p, info);
  PSOCI_HIP(hipGetLastError());
  c.sync();
  // the blocks' kept elements
  const int64_t nbatch = (nstage + kBatch - 1) / kBatch;
  const size_t nwords = (size_t)(nstage + 63) / 64;
  Scratch sb{c.spare.buf[1]};
  sb.buf.reserve(sb.bytes(nstage, 8) + 2 * sb.bytes(nwords + 2, 8) + sb.bytes(nwords, 2) + sb.bytes(nbatch, 8) +
               sb.bytes(n, 8) + sb.bytes(n, 4));
  double* staging = sb.take<double>(nstage);
  uint64_t* bits = sb.take<uint64_t>(nwords + 2);
  uint64_t* tbits = sb.take<uint64_t>(nwords + 2);
  uint16_t* rank = sb.take<uint16_t>(nwords);
  int64_t* first = sb.take<int64_t>(nbatch);
  uint64_t* amask = sb.take<uint64_t>(n);
  int32_t* cfg = sb.take<int32_t>(n);
  hipLaunchKernelGGL(k_sef_masks, dim3(per_cfg), dim3(256), 0, c.stream, ncfg, c.d_dm.p, c.d_sm.p, c.d_nopen.p,
                     c.d_pat.p, c.d_patoff.p, c.d_cls.p, c.d_nsef.p, c.d_sefoff.p, sp.frac ? 1 : 0, amask, cfg);
  PSOCI_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_batch_first, dim3(blocks_for(np, 256)), dim3(256), 0, c.stream, np, boff, first);
  PSOCI_HIP(hipGetLastError());
  // a wavefront per batch
  hipLaunchKernelGGL(sp.frac ? k_block_elems<true> : k_block_elems<false>, dim3(blocks_for(nbatch, 4)), dim3(256), 0,
                     c.stream, nstage, np, boff, first, info, c.d_dm.p, c.d_sm.p, c.d_nopen.p, c.d_cph.p, c.d_cmult.p,
                     c.d_nsef.p, c.d_sefoff.p, amask, c.d_two.p, staging, bits, rank);
  PSOCI_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_transpose_bits, dim3(blocks_for(nbatch, 4)), dim3(256), 0, c.stream, nstage, np, boff, first,
                     info, c.d_nsef.p, bits, tbits);
  PSOCI_HIP(hipGetLastError());
  // the rows: counts, offsets, elements
  hipLaunchKernelGGL(k_segs, dim3((unsigned)ncfg), dim3(256), 0, c.stream, ncfg, off.p, list, info, boff, c.d_nsef.p,
                     c.d_sefoff.p, segs);
  PSOCI_HIP(hipGetLastError());
  PSOCI_HIP(hipMemsetAsync(cnt.p + n, 0, sizeof(int64_t), c.stream));
  // a wavefront per row, in whole groups of 8 x 16 workgroups
  const unsigned per_row = (blocks_for(n, 4) + 127) / 128 * 128;
  hipLaunchKernelGGL(k_rows<false>, dim3(per_row), dim3(256), 0, c.stream, n, ncfg, cfg, off.p, c.d_nsef.p,
                     c.d_sefoff.p, segs, bits, tbits, rank, staging, cnt.p, nullptr, nullptr, nullptr, nullptr, nullptr,
                     nullptr);
  PSOCI_HIP(hipGetLastError());
  c.d_rowptr.alloc(n + 1);
  c.scan(cnt.p, c.d_rowptr.p, n + 1);
  int64_t nnz = 0;
  PSOCI_HIP(hipMemcpyAsync(&nnz, c.d_rowptr.p + n, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
  c.sync();
  c.d_col.alloc(nnz);
  c.d_val.alloc(nnz);
  c.d_val32.alloc(nnz);
  c.d_lowcnt.alloc(n);
  c.d_diag.alloc(n);
  hipLaunchKernelGGL(k_rows<true>, dim3(per_row), dim3(256), 0, c.stream, n, ncfg, cfg, off.p, c.d_nsef.p,
                     c.d_sefoff.p, segs, bits, tbits, rank, staging, nullptr, c.d_rowptr.p, c.d_col.p, c.d_val.p,
                     c.d_val32.p, c.d_lowcnt.p, c.d_diag.p);
  PSOCI_HIP(hipGetLastError());
  // the reference's element count: the lower parts
  c.nnz_full = nnz;
  c.nnz_lower = (nnz + n) / 2;
  c.sync();
  c.have_h = true;
  const auto t1 = std::chrono::steady_clock::now();
  tune_stored(c);
  c.have_diag = true;
  c.hbuild_seconds[0] = std::chrono::duration<double>(t1 - t0).count();
  c.hbuild_seconds[1] = std::chrono::duration<double>(std::chrono::steady_clock::now() - t1).count();
}

void compute_diag(Ctx& c) {
  const Space& sp = c.sp;
  c.d_diag.alloc(sp.nsef_total);
  hipLaunchKernelGGL(k_diag_only, dim3(blocks_for(sp.ncfg, 4)), dim3(256), 0, c.stream, sp.ncfg, c.d_dm.p, c.d_sm.p,
                     c.d_nopen.p, c.d_cph.p, c.d_pat.p, c.d_patoff.p, c.d_cls.p, c.d_cmult.p, c.d_nsef.p,
                     c.d_sefoff.p, sp.nbf, sp.frac ? 1 : 0, c.d_one.p, c.d_two.p, c.d_diag.p);
  PSOCI_HIP(hipGetLastError());
  c.sync();
  c.have_diag = true;
}

void block_on_device(Ctx& c, int64_t I, int64_t J, double* host_out, int* status) {
  const Space& sp = c.sp;
  int ni = sp.nsef[I], nj = sp.nsef[J];
  DevBuf<double> out;
  DevBuf<PairInfo> P;
  out.alloc((size_t)ni * nj);
  P.alloc(1);
  hipLaunchKernelGGL(k_single_block, dim3(1), dim3(256), 0, c.stream, P.p, (int)I, (int)J, c.d_dm.p, c.d_sm.p,
                     c.d_nopen.p, c.d_cph.p, c.d_pat.p, c.d_patoff.p, c.d_cls.p, c.d_cmult.p, c.d_jsym.p,
                     c.d_nsef.p, sp.nbf, sp.frac ? 1 : 0, c.d_one.p, c.d_two.p, out.p);
  PSOCI_HIP(hipGetLastError());
  PairInfo hp;
  out.download(host_out, (size_t)ni * nj, c.stream);
  P.download(&hp, 1, c.stream);
  c.sync();
  if (status) *status = hp.kind != 0 ? 1 : 0;
}

void get_h_lower(Ctx& c, int64_t* rowptr, int32_t* col, double* val, double* diag) {
  const int64_t n = c.sp.nsef_total;
  std::vector<int32_t> lc(n);
  c.d_lowcnt.download(lc.data(), n, c.stream);
  c.sync();
  std::vector<int64_t> lp(n + 1);
  int64_t acc = 0;
  for (int64_t r = 0; r < n; ++r) {
    lp[r] = acc;
    acc += lc[r];
  }
  lp[n] = acc;
  if (rowptr) std::copy(lp.begin(), lp.end(), rowptr);
  if (col || val) {
    DevBuf<int64_t> d_lp;
    DevBuf<int32_t> lcol;
    DevBuf<double> lval;
    d_lp.upload(lp, c.stream);
    lcol.alloc(acc);
    lval.alloc(acc);
    hipLaunchKernelGGL(k_extract_lower, dim3(blocks_for(n, 4)), dim3(256), 0, c.stream, n, c.d_rowptr.p,
                       c.d_lowcnt.p, d_lp.p, c.d_col.p, c.d_val.p, lcol.p, lval.p);
    PSOCI_HIP(hipGetLastError());
    if (col) lcol.download(col, acc, c.stream);
    if (val) lval.download(val, acc, c.stream);
    c.sync();
  }
  if (diag) {
    c.d_diag.download(diag, n, c.stream);
    c.sync();
  }
}

void install_h(Ctx& c, const std::vector<int64_t>& rowptr, const std::vector<int32_t>& col,
               const std::vector<double>& val, const std::vector<int32_t>& lowcnt, const std::vector<double>& diag) {
  const int64_t n = c.sp.nsef_total, nnz = rowptr[n];
  c.have_h = false;
  c.d_rowptr.upload(rowptr, c.stream);
  c.d_col.upload(col, c.stream);
  c.d_val.upload(val, c.stream);
  c.d_lowcnt.upload(lowcnt, c.stream);
  c.d_diag.upload(diag, c.stream);
  c.d_val32.alloc(nnz);
  if (nnz > 0)
    hipLaunchKernelGGL(k_to_f32, dim3(blocks_for(nnz, 256)), dim3(256), 0, c.stream, nnz, c.d_val.p, c.d_val32.p);
  PSOCI_HIP(hipGetLastError());
  c.nnz_full = nnz;
  c.nnz_lower = (nnz + n) / 2;
  c.sync();
  c.have_h = true;
  c.have_diag = true;
  c.hbuild_seconds[0] = c.hbuild_seconds[1] = -1.0;  // not built here
}

}  // namespace psoci
