// Context state of the PSOCI MI355X library (one GPU).
#pragma once
#include "common.hpp"
#include "linalg.hpp"
#include "elem.hpp"
#include "ras.hpp"

namespace psoci {

constexpr int kSpmmBuckets = 5;  // row-length classes of the stored sigma

// Caller-provided device memory for the padded column staging of a sigma
// call (p null: the context's own buffer, grown on demand).
struct Staging {
  void* p = nullptr;
  size_t bytes = 0;
};

// Scratch memory of the Hamiltonian build (buf 0, 1), of the Davidson solver (2)
// and of the adjoint (3), kept for the context's next one (new integrals at the
// next geometry): allocating and freeing it every time cost 0.5 ms beside a 1.6
// ms build (32,000 SEFs, 0.85 GB), and 20 ms where several contexts built in
// turn.  A context keeps up to kSpareBytes in all and, beyond a sixteenth of
// that, no more than a sixteenth of the device memory that is free when it grows
// (asking every time cost 10 us).  Given back when an allocation of any context
// on the device fails, before the direct engine sizes its plan, and with the
// context.
constexpr size_t kSpareBytes = size_t(1) << 30;
struct Spare {
  DevBuf<char> buf[4];
  int device = -1;  // of the context
  size_t allowed = kSpareBytes / 16;  // what it may keep without asking
  bool busy[4] = {false, false, false, false};  // in use by a scope of the context's thread
  Spare();
  ~Spare();
  Spare(const Spare&) = delete;
  Spare& operator=(const Spare&) = delete;
  bool give_back();  // frees what no scope uses; whether there was any
  void take(int first, int count);
  void leave(int first, int count);
};
// The buffers first .. first + count - 1 in use by a scope; the stream is idle
// where it ends normally.
struct SpareUse {
  Spare& s;
  const int first, count;
  SpareUse(Spare& s_, int first_, int count_) : s(s_), first(first_), count(count_) { s.take(first, count); }
  SpareUse(const SpareUse&) = delete;
  SpareUse& operator=(const SpareUse&) = delete;
  ~SpareUse() { s.leave(first, count); }
};
// Arrays carved from one of the spare buffers.
struct Scratch {
  DevBuf<char>& buf;
  size_t used = 0;
  static constexpr size_t bytes(size_t count, size_t size) { return (count * size + 255) / 256 * 256; }
  template <typename T>
  T* take(size_t count) {
    T* p = reinterpret_cast<T*>(buf.p + used);
    used += bytes(count, sizeof(T));
    return p;
  }
};
inline thread_local Spare* t_spare = nullptr;  // of the context whose entry point runs on this thread

struct Ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;

  Space sp;
  bool have_space = false;
  int nbf_ints = 0;
  double ecore = 0.0;
  bool have_ints = false;
  // fingerprints of the inputs (configuration list, integrals), written into
  // a stored-Hamiltonian checkpoint and checked when one is loaded
  uint64_t space_hash = 0, ints_hash = 0;

  // space on the device
  DevBuf<uint64_t> d_dm, d_sm;
  DevBuf<int8_t> d_nopen;
  DevBuf<int32_t> d_nsef;
  DevBuf<int64_t> d_sefoff;
  DevBuf<uint8_t> d_cph;
  DevBuf<uint16_t> d_pat;
  DevBuf<int32_t> d_patoff;    // 24: two pattern families
  DevBuf<uint8_t> d_cls;       // per configuration: pattern family
  DevBuf<double> d_cmult;      // per configuration: SEF combination sign
  DevBuf<int32_t> d_jsym;      // per configuration
  DevBuf<double> d_one, d_two;

  // stored Hamiltonian: symmetric full CSR (lower part first in each row)
  bool have_h = false;
  int64_t nnz_lower = 0, nnz_full = 0;
  DevBuf<int64_t> d_rowptr;   // full, n+1
  DevBuf<int32_t> d_col;      // full
  DevBuf<double> d_val;       // full FP64
  DevBuf<float> d_val32;      // full FP32
  DevBuf<int32_t> d_lowcnt;   // per row: entries of the lower part (incl. diagonal)
  // stored sigma shape per precision ([0] FP64, [1] FP32) at 16 columns:
  // lanes per nonzero, rows per wavefront (spmm_fixed: for every width)
  bool spmm_fixed[2] = {false, false};
  int units = 0;  // compute units of the device
  int spmm_g[2] = {1, 1}, spmm_r[2] = {1, 1};
  double spmm_tune_ms[2] = {-1, -1};
  // row-length buckets (kSpmmBuckets length classes): the rows of each in
  // d_brows[spmm_boff[b] .. spmm_boff[b + 1]), a shape per bucket and
  // precision, and whether the bucketed launches are used (count_buckets and
  // tune_stored in sigma.hip)
  DevBuf<int32_t> d_brows;
  int64_t spmm_boff[kSpmmBuckets + 1] = {0};  // rows before each
  int spmm_bg[2][kSpmmBuckets] = {}, spmm_br[2][kSpmmBuckets] = {};
  bool spmm_bucketed[2] = {false, false};
  double hbuild_seconds[2] = {-1.0, -1.0};  // last build_h: build proper, shape tuner
  double spmm_bucket_ms[2] = {-1, -1};
  DevBuf<double> d_diag;
  bool have_diag = false;

  // direct sigma: every connected configuration (both directions, J = I
  // included) per configuration I, ascending, and per-determinant alpha
  // open-shell masks
  bool have_pairs = false;
  int64_t nadj = 0;
  int64_t direct_elems = 0;  // structural SEF elements per direct sigma
  int64_t direct_det_pairs = -1;  // connected determinant pairs per direct sigma (-1: not counted yet)
  DevBuf<int64_t> d_adjoff;   // ncfg + 1: first record of each configuration
  DevBuf<PairRec> d_rec;      // one record per ordered connected pair
  DevBuf<double> d_cdiag;     // ncfg: vnt[0] of each diagonal block
  DevBuf<int32_t> d_ndbl;     // ncfg: double-excitation records (first in each segment)
  DevBuf<int32_t> d_nsgl;     // ncfg: single-excitation records (next)
  DevBuf<int32_t> d_order;    // alternative row order of the direct sigma (items when split)
  DevBuf<int32_t> d_items;    // split spaces: the natural order's work items
  // schedule of the direct sigma per precision ([0] FP64, [1] FP32)
  bool direct_order[2] = {false, false};  // use d_order
  bool direct_split = false;  // rows are work items (I << 2 | q): SEFs [64q, 64q + 64) of I
  int64_t direct_nrows = 0;   // rows (work items) per direct sigma launch
  int direct_chunk[2] = {0, 0};         // XCD run length (workgroups)
  double direct_tune_ms[2] = {-1, -1};  // the tuner's best sample time (-1: fixed by the environment)
  DevBuf<ConfRec> d_conf;     // packed configurations
  DevBuf<double> d_xt;        // XT[e][f][o] = (e o|o f)
  DevBuf<int64_t> d_detoff;   // ncfg
  DevBuf<uint64_t> d_detao;   // ndet_total
  DevBuf<int16_t> d_didx;     // determinant index by open-shell pattern (Space::didx)

  // direct sigma engine: requested (0 auto: the string-driven one where the
  // space qualifies, else the configuration records; 1 configuration
  // records; 2 string-driven only) and the string-driven plan (strsig.hip)
  int direct_engine_req = 0;
  // (two parts, each tried once: the strings, which the adjoint needs too,
  // and the products)
  bool have_strings = false, strings_tried = false;
  bool have_ras = false, ras_tried = false;
  std::string ras_why;
  bool zero_integral = false;  // a two-electron integral is exactly zero
  RasPlan ras;
  DevBuf<uint64_t> d_rasmask;
  DevBuf<int8_t> d_rascls;
  DevBuf<uint32_t> d_rasadd;
  DevBuf<int32_t> d_rasrem;
  DevBuf<RasBlockDev> d_rasblk;
  DevBuf<RasCmp> d_rascmp;
  DevBuf<int16_t> d_rasq, d_raspidx;
  DevBuf<RasTile> d_rastile[4];        // product tiles for chunks of 16, 8, 4 and 2 columns
  std::vector<RasLaunch> ras_launch[4];  // and their launches
  DevBuf<RasSef> d_rassef;
  DevBuf<double> d_rasg64;  // the compact products' matrices
  DevBuf<float> d_rasg32;
  DevBuf<RasView> d_rasview;
  DevBuf<char> d_rasc, d_rasw;  // determinant vectors [2 ndet + 1][16 FP32 | ras_kc64 FP64], W [cwunit][same]
  int ras_kc64 = 8;             // FP64 columns per chunk (16 when memory allows, else 8)
  DevBuf<int32_t> d_rasdidx;    // [cdunit]: signed vector row (det + negative * ndet) of every D entry
  DevBuf<int64_t> d_rastoff;    // nsef + 1: first term of each SEF
  int64_t ras_nterm = 0;        // terms over all SEFs (after merging mirrored pairs)
  DevBuf<int32_t> d_rasterm;    // signed W offsets (bit 31: negative)
  DevBuf<int8_t> d_rasscl;      // per SEF: 0 1/sqrt(2), 1 sqrt(2), 2 one
  DevBuf<int32_t> d_rasabsent;  // determinants of no SEF (a list that is part of its space)
  DevBuf<int32_t> d_rasorder;   // the order the SEFs are walked in (d_rastoff, d_rasscl, d_rasrows follow it)
  DevBuf<int2> d_rasrows;       // per SEF: signed rows of its determinants' coefficients
  // the string-driven adjoint (rasrdm.hip): whether it equals the pair walk
  // (no integral sum that the reference's blocks leave out)
  bool ras_rdm = false;
  void drop_products() {
    have_ras = false;
    d_rascmp.release();
    for (int k = 0; k < 4; ++k) {
      d_rastile[k].release();
      ras_launch[k].clear();
    }
    d_rasg64.release();
    d_rasg32.release();
    d_rasw.release();
    d_rasdidx.release();
    d_rastoff.release();
    d_rasterm.release();
    d_rasscl.release();
  }
  // everything built; what has been tried stays so
  void drop_plan() {
    drop_products();
    have_strings = ras_rdm = false;
    ras = RasPlan();
    d_rasmask.release();
    d_rascls.release();
    d_rasadd.release();
    d_rasrem.release();
    d_rasblk.release();
    d_rasq.release();
    d_raspidx.release();
    d_rassef.release();
    d_rasview.release();
    d_rasc.release();
    d_rasrows.release();
    d_rasorder.release();
    d_rasabsent.release();
  }
  void drop_ras() {
    drop_plan();
    strings_tried = ras_tried = false;
  }

  // transition Hamiltonian (rows: this list's SEFs; columns: a second
  // list's SEFs placed at this list's entry points), lower by index
  bool have_trans = false;
  int64_t nnz_trans = 0;
  DevBuf<int64_t> d_trow;
  DevBuf<int32_t> d_tcol;
  DevBuf<double> d_tval;

  // scratch
  DevBuf<char> d_pad;  // zero-padded column staging for the direct sigma
  Spare spare;
  LinalgHost lin_host;  // the Davidson's small matrices
  void* scan_tmp = nullptr;
  size_t scan_tmp_bytes = 0;

  ~Ctx() {
    if (scan_tmp) (void)hipFree(scan_tmp);
    if (stream) (void)hipStreamDestroy(stream);
  }
  void scan(const int64_t* in, int64_t* out, int64_t n) { exclusive_scan_i64(in, out, n, stream, scan_tmp, scan_tmp_bytes); }
  void sync() { PSOCI_HIP(hipStreamSynchronize(stream)); }
};

// kernels-side entry points (hbuild.hip, sigma.hip, ...)
void upload_space(Ctx& c);
void build_pairs(Ctx& c);               // adjacency + determinant masks (direct sigma, adjoint)
void build_h(Ctx& c);                   // stored Hamiltonian
// a checkpoint's stored-sigma choices per precision: whether rows are launched
// by length class (chosen: the writer chose by the present rule), and the
// shapes where the writer had fixed them
struct SpmmSaved {
  bool fixed[2], chosen[2], bucketed[2];
  int g[2], r[2], bg[2][kSpmmBuckets], br[2][kSpmmBuckets];
};
// the stored sigma's shapes and row-length buckets (after build_h or a load)
void tune_stored(Ctx& c, const SpmmSaved* saved = nullptr);
void compute_diag(Ctx& c);              // diagonal only
void block_on_device(Ctx& c, int64_t I, int64_t J, double* host_out, int* status);
void sigma_stored(Ctx& c, int prec, int k, const void* X, int ldx, void* Y, int ldy, const Staging& st = Staging{});
void sigma_direct(Ctx& c, int prec, int k, const void* X, int ldx, void* Y, int ldy, const Staging& st = Staging{});
int64_t direct_det_pairs(Ctx& c);
// string-driven direct sigma (strsig.hip): the plan's strings (adjoint: only
// where they serve the adjoint) and its products (false when the space does
// not qualify; c.ras_why says why), and the sigma
bool build_strings(Ctx& c, bool adjoint);
bool build_ras(Ctx& c);
void sigma_ras(Ctx& c, int prec, int k, const void* X, int ldx, void* Y, int ldy);
// columns [col0, col0 + kw) of X [n][ldx] as FP64 determinant vectors in
// c.d_rasc; returns their padded width
inline int ras_width64(int kw) { return kw > 8 ? 16 : kw > 4 ? 8 : kw > 2 ? 4 : 2; }
int ras_scatter64(Ctx& c, const double* X, int ldx, int col0, int kw);
// the adjoint through the string plan (needs have_strings and ras_rdm)
void ras_rdm_grad(Ctx& c, int k, const double* dC, const double* w, double* d_g1, double* d_g2);
// one timed sigma of k columns on internal buffers, averaged over reps: ms[5]
// per launch group (scatter, products by kind, gather), flops[3] per kind
void ras_timing(Ctx& c, int prec, int k, int reps, double* ms, double* flops);
// the direct sigma's operator: the string-driven plan where requested and
// possible, else the configuration pair records (throws when engine 2 is
// requested and the space does not qualify)
void build_direct(Ctx& c);
// the engine a direct sigma uses with what is built now (0: none yet)
inline int direct_engine(const Ctx& c) {
  // (a plan of the automatic choice's wider spaces does not serve a request)
  const bool wide = c.ras.fill < 1.0 || c.ras.frac;
  if (c.have_ras && (c.direct_engine_req == 0 || (c.direct_engine_req == 2 && !wide))) return 2;
  if (c.direct_engine_req != 2 && c.have_pairs) return 1;
  return 0;
}
// whether build_direct would build something (the string plan not tried yet
// where it may apply, or no operator at all)
inline bool direct_needs_build(const Ctx& c) {
  if (c.direct_engine_req != 1 && !c.have_ras && !c.ras_tried) return true;
  return direct_engine(c) == 0;
}  // connected determinant pairs per direct sigma (one counting launch, cached)
// staging bytes a sigma call of k columns at strides ldx, ldy needs (0: none)
size_t sigma_staging_bytes(const Ctx& c, int mode, int prec, int k, const void* X, int ldx, const void* Y, int ldy);
// the allocation-free scratch array of the current device (noalloc.hip):
// set up once per device by psoci_ctx_create, then its address and size
int noalloc_init(int device);
void noalloc_scratch(int device, void** p, size_t* bytes);
void get_h_lower(Ctx& c, int64_t* rowptr, int32_t* col, double* val, double* diag);
// installs a stored Hamiltonian given as the full symmetric CSR (lower part
// first in each row, lowcnt entries) and its diagonal (restart.cpp -> hbuild.hip)
void install_h(Ctx& c, const std::vector<int64_t>& rowptr, const std::vector<int32_t>& col,
               const std::vector<double>& val, const std::vector<int32_t>& lowcnt, const std::vector<double>& diag);
// per-configuration energy contributions of k roots (analysis.hip)
void energy_contrib(Ctx& c, int k, const double* dC, const double* d_evals, double* d_deltae);
void save_h(Ctx& c, const char* path);  // stored-Hamiltonian checkpoint (restart.cpp)
void load_h(Ctx& c, const char* path);
void rdm_grad(Ctx& c, int k, const double* dC, const double* w, double* d_g1, double* d_g2);
void build_transition(Ctx& c, const Space& list2, int64_t* nnz);  // transition.hip

struct DavParams;
int davidson(Ctx& c, const psoci_dav_params& p, double* evals, double* evecs, psoci_dav_stats* st);

inline ConfView conf_view_host(const Space& sp, int64_t c, const uint16_t* pat_dev) {
  ConfView v;
  v.d = sp.dm[c];
  v.s = sp.sm[c];
  v.nopen = sp.nopen[c];
  v.ph = sp.cphase[c];
  v.pat = pat_dev + sp.pat_off[12 * sp.cls[c] + v.nopen];
  return v;
}

}  // namespace psoci
