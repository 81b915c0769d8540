// Single-network engine (device buffers, launch sequences, hipGraph of one /
// eight DP45 attempts, output rings) shared by the per-precision
// translation units kmt_engine_f32.hip / kmt_engine_f64.hip; the C ABI in
// kmt_api.hip reaches it through EngineBase.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/kuramoto_amd.h"
#include "kmt_common.hpp"
#include "kmt_kernels.hpp"
#include "kmt_sign.hpp"
#include "kmt_sym.hpp"

namespace kmt {

#define fail kmt_fail

static inline long round_up(long x, long m) { return (x + m - 1) / m * m; }

// ---------------------------------------------------------------------
// Engine
// ---------------------------------------------------------------------
struct EngineBase {
  virtual ~EngineBase() {}
  virtual int create(int, long, double, double, int, double) = 0;
  virtual int set_omega(const void *) = 0;
  virtual int set_state(const void *, double, double) = 0;
  virtual int get_state(void *, double *, double *) = 0;
  virtual int set_adjacency(const void *, int, long, int) = 0;
  virtual int set_factor(const void *, const void *, int) = 0;
  virtual int set_factor_sign(int, uint32_t) = 0;
  virtual int build_adjacency(int) = 0;
  virtual int use_factored(int) = 0;
  virtual int get_adjacency_rows(long, long, void *) = 0;
  virtual int rhs(const void *, void *, void *) = 0;
  virtual int rhs_device(const void *, void *, void *, void *, hipStream_t) = 0;
  virtual size_t rhs_scratch_bytes() const = 0;
  virtual int device_index() const = 0;
  virtual int order(const void *, double *) = 0;
  virtual int begin(const double *, int, double, int, int) = 0;
  virtual int advance(int, kmt_status *) = 0;
  virtual int read_outputs(int, void *, void *, void *, int *) = 0;
  virtual int read_times(int, void *, void *, int *) = 0;
  virtual int step(int *, double *, double *) = 0;
  virtual int eval(double, void *) = 0;
  virtual int time_stage(int, double *) = 0;
  virtual int time_attempts(int, double *, double *, kmt_status *) = 0;
  virtual int layout(long *, int *, int *, int *) = 0;
  virtual int tune(int, double *) = 0;
  virtual int select_variant(int, int) = 0;
  double mscale_ = 1.0;
};

template <class R> struct Engine : EngineBase {
  int device = 0;
  long N = 0, ldv = 0, rows_alloc = 0, lda = 0;
  R atl = 0, rtl = 0, c1 = 0;
  int fixed = 0;
  hipStream_t stream = nullptr;

  // vectors (ldv each unless noted)
  R *y = nullptr, *ylast = nullptr, *ynew = nullptr, *omega = nullptr, *kbuf = nullptr, *k[7] = {};
  R *cs[2] = {nullptr, nullptr};  // 2*ldv each
  R *cs_scr = nullptr, *vec_scr = nullptr, *f_scr = nullptr, *pairs = nullptr, *k_scr = nullptr;  // scratch
  double *err_part = nullptr;
  int n_err_part = 0;
  double *ord_scr = nullptr;  // stand-alone order parameter partials + result
  State<R> *st = nullptr;
  State<R> *st_host = nullptr;  // pinned
  // Host copy of the device state.  fresh: equal to it up to the host's own
  // drains (nothing launched since it was fetched), so reading entry points
  // need no round trip; dirty: drains not yet sent, written back before the
  // next launch that uses the state.
  State<R> shadow{};
  bool fresh = false, dirty = false;
  // pinned staging of row drains (two halves, grown to at most kStageMax each)
  static constexpr size_t kStageMax = (size_t)1 << 20;
  char *stage_buf = nullptr;
  size_t stage_half = 0;
  hipEvent_t stage_ev[2] = {nullptr, nullptr};

  // adjacency
  int storage = -1;  // KMT_ADJ_*
  void *A = nullptr;
  size_t A_bytes = 0;
  R *X = nullptr, *w = nullptr;
  R *XT = nullptr;  // transposed factor [K][ldv] (K <= kLrMaxRank): the low-rank and register-rebuild forms
  int K = 0;
  int factored = 0;  // 0 dense A, KMT_LOWRANK_CONTRACT, KMT_LOWRANK_REBUILD
  // KMT_ADJ_SYM: (I, J) of each stored block, and the row / column partials
  long sym_nb = 0, sym_blocks = 0;
  int2 *sym_ij = nullptr;
  SymPair<double> *sym_prow = nullptr, *sym_pcol = nullptr;
  double *lr_part = nullptr, *lr_G = nullptr;
  int lr_nblk = 0, lr_blocks = 0;
  // packed +-1 factor (kmt_set_factor_sign): per pass (1: rows m over
  // k = n, 2: rows n over k = m) the sign bits in the pass's tile order
  // (ldp rows of 32 npairs words: the bit rows, the ones row, zero rows),
  // the B fragments of the digits and the int32 partial sums
  int sign = 0;
  struct SignPass {
    long ldp = 0, nsb = 0, npairs = 0;  // nsb = 2 npairs super-blocks of 512
    long units = 1;       // row groups of 256 x pairs
    int wgs = 1;          // workgroups that share the units
    int nsplit = 1;       // most workgroups of one row group: slots of part
    uint32_t *tiles = nullptr;
    uint8_t *bfrag = nullptr;      // owns bfrag_rhs and part too
    uint8_t *bfrag_rhs = nullptr;  // pass 1: the vector of a stand-alone right-hand side
    int32_t *part = nullptr;
    uint32_t *ones = nullptr;  // the ones row: bits set for k < kdim, 16 nsb words
  } s_pass[2];
  std::vector<R> X_host, w_host;

  // run
  int begun = 0;
  R *t_eval = nullptr;
  int n_eval = 0;
  R *ring = nullptr, *r_ring = nullptr, *times = nullptr;
  double *ord_part = nullptr;
  int ring_cap = 0, keep_rows = 0, times_cap = 4096, nblk_emit = 0;
  hipGraphExec_t g1 = nullptr, g8 = nullptr;
  bool graphs_valid = false;
  int tune_rows = 8, tune_nt = 1, tune_bal = 0, tune_ring = 0, tuned = 0;
  int pinned = 0;  // attempts follow a variant chosen by the caller (kmt_select_variant) or timed (kmt_autotune)
  double tune_ms[12] = {0};
  int bal_grid = 0;  // workgroups of the balanced variant (one resident round)
  R t0_ = 0, h0_ = 0;

  ~Engine() override { release(); }

  void release() {
    if (stream) (void)hipStreamSynchronize(stream);
    drop_graphs();
    R *vecs[] = {y, ylast, ynew, omega, kbuf, cs[0], cs[1], cs_scr, vec_scr, f_scr, pairs, k_scr, X, w, XT, t_eval, ring, r_ring, times};
    for (R *p : vecs)
      if (p) (void)hipFree(p);
    double *dv[] = {err_part, ord_scr, lr_part, lr_G, ord_part};
    drop_sign();
    for (double *p : dv)
      if (p) (void)hipFree(p);
    if (st) (void)hipFree(st);
    if (sym_ij) (void)hipFree(sym_ij);
    if (sym_prow) (void)hipFree(sym_prow);
    if (sym_pcol) (void)hipFree(sym_pcol);
    if (st_host) (void)hipHostFree(st_host);
    if (stage_buf) (void)hipHostFree(stage_buf);
    for (hipEvent_t e : stage_ev)
      if (e) (void)hipEventDestroy(e);
    if (A) (void)hipFree(A);
    if (stream) (void)hipStreamDestroy(stream);
    y = ylast = ynew = omega = kbuf = nullptr;
    stream = nullptr;
  }

  // Destroy the captured attempt graphs.  Every entry point that launches
  // them synchronises the stream before it returns, so none is in flight
  // here; the synchronisation keeps that true for any later caller.
  void drop_graphs() {
    if ((g1 || g8) && stream) (void)hipStreamSynchronize(stream);
    if (g1) (void)hipGraphExecDestroy(g1);
    if (g8) (void)hipGraphExecDestroy(g8);
    g1 = g8 = nullptr;
    graphs_valid = false;
  }

  int alloc_vec(R **p, long n) {
    HIP_TRY(hipMalloc((void **)p, sizeof(R) * n));
    HIP_TRY(hipMemsetAsync(*p, 0, sizeof(R) * n, stream));
    return KMT_OK;
  }

  int create(int dev, long n, double a, double r, int fx, double c) override {
    device = dev;
    N = n;
    atl = (R)a;
    rtl = (R)r;
    fixed = fx;
    c1 = (R)c;
    HIP_TRY(hipSetDevice(device));
    HIP_TRY(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    ldv = round_up(N, 64);
    lda = ldv;
    rows_alloc = round_up(N, 64);
    KMT_TRY(alloc_vec(&y, ldv));
    KMT_TRY(alloc_vec(&ylast, ldv));
    KMT_TRY(alloc_vec(&ynew, ldv));
    KMT_TRY(alloc_vec(&omega, ldv));
    KMT_TRY(alloc_vec(&kbuf, 7 * ldv));
    for (int j = 0; j < 7; ++j) k[j] = kbuf + j * ldv;
    KMT_TRY(alloc_vec(&cs[0], 2 * ldv));
    KMT_TRY(alloc_vec(&cs[1], 2 * ldv));
    KMT_TRY(alloc_vec(&cs_scr, 2 * ldv));
    KMT_TRY(alloc_vec(&vec_scr, ldv));
    KMT_TRY(alloc_vec(&f_scr, ldv));
    KMT_TRY(alloc_vec(&pairs, 2 * ldv));
    // one error partial per stage-7 workgroup: at most one per row (every
    // grid - row groups, balanced, low-rank, rebuilt rows - has <= N workgroups)
    n_err_part = (int)rows_alloc;
    HIP_TRY(hipMalloc((void **)&err_part, sizeof(double) * n_err_part));
    HIP_TRY(hipMalloc((void **)&ord_scr, sizeof(double) * (2 * ((ldv + kBlock - 1) / kBlock) + 2)));
    HIP_TRY(hipMalloc((void **)&st, sizeof(State<R>)));
    HIP_TRY(hipHostMalloc((void **)&st_host, sizeof(State<R>), hipHostMallocDefault));
    std::memset(&shadow, 0, sizeof(shadow));
    shadow.atl = atl;
    shadow.rtl = rtl;
    shadow.fixed = fixed;
    shadow.times_cap = times_cap;
    HIP_TRY(hipMemcpyAsync(st, &shadow, sizeof(shadow), hipMemcpyHostToDevice, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  int layout(long *plda, int *eb, int *rows, int *flags) override {
    if (plda) *plda = sym() ? kSymT : lda;
    if (eb) *eb = storage < 0 ? (int)sizeof(R) : (int)elem_bytes(storage);
    if (rows) *rows = tune_rows;
    if (flags) *flags = (tune_nt ? 1 : 0) | (tune_bal ? 2 : 0) | (tune_ring ? 4 : 0);
    return KMT_OK;
  }
  // The stage-7 error partials are summed per workgroup, so their grouping,
  // and with it the last bits of the error norm and of h, follows the rows of
  // stage 7's variant.  Those are a rule of their own (error_rows) that says
  // nothing about speed, and every choice is by a fixed rule, not by timing,
  // so that runs and restarts of one problem give the same bits in every
  // context and process.  The other stages write no partials and sum every
  // row in the same order in every variant:
  //  * A matrix that fits the 256 MB Infinity Cache is read from it by every
  //    stage after the first, so its loads are plain (a non-temporal load
  //    does not keep the line: FP64 N=5000, 200 MB, 34.8 -> 30.6 us; FP32
  //    N=8000, 256 MB, 40.6 -> 38.1; BF16 N=11000, 242 MB, 43.6 -> 36.7; from
  //    484 MB on plain loads lose: FP32 N=11000 83.8 against 74.0), and from
  //    N = 4096 on it takes 4 rows per group, which fills the chip at N=5000
  //    (17.8 against 18.2 us with 8 rows, 20.9 with 16).  With FP64 vectors
  //    and 16-bit entries 8 rows: the vectors' bytes are then no more than the
  //    entries' (BF16 N=8000: 26.1 us against 30.7 with 4 rows).  Smaller N
  //    keep 8 rows.
  //  * A larger one takes 8 rows with non-temporal loads, 16 rows with 16-bit
  //    entries (each (cos, sin) chunk is reused for every row of the group:
  //    FP64 state, BF16, N=50000: 0.752 against 0.812 ms with 8 rows; FP32
  //    state, FP16, N=200000: 11.4 against 12.0), but 8 with FP32 vectors
  //    below N = 50000, where the vectors are small and the shorter groups end
  //    more evenly (BF16 N=14000: 62.8 against 65.2 us; N=50000: level).
  //  * The chunk ring wherever it measured faster: the working precision
  //    (0.6% at N=50000, 2-4% from the cache) and 16-bit entries with FP32
  //    vectors from the cache (5%); with 16 rows of 16-bit entries it needs
  //    231 registers and is 5% slower.
  // kmt_autotune / kmt_select_variant override it.
  void default_variant() {
    const bool half = elem_bytes(storage) == 2;
    const bool cached = (double)N * (double)N * (double)elem_bytes(storage) <= 256e6;
    tune_rows = !cached ? (half && (sizeof(R) == 8 || N >= 50000) ? 16 : 8) : N < 4096 || (half && sizeof(R) == 8) ? 8 : 4;
    tune_nt = cached ? 0 : 1;
    tune_bal = 0;
    tune_ring = !half || (cached && sizeof(R) == 4);
    bal_grid = 0;
    tuned = 1;
    drop_graphs();
  }

  // Rows per error partial.  16-bit entries: 16; the working precision: 8 (the
  // grouping of the FP64 register-rebuild kernel for K <= 8, whose runs are
  // the dense ones' bit for bit); 4 from N = 4096 on up to 128 MB.  Any fixed
  // choice would do; another one is another sequence of steps.
  int error_rows() const {
    if (pinned) return tune_rows;
    if (N >= 4096 && (double)N * (double)N * (double)elem_bytes(storage) <= 128e6) return 4;
    return elem_bytes(storage) == 2 ? 16 : 8;
  }

  // Every entry point that launches the dense kernel uses the rule's choice:
  // a right-hand side evaluated before any run too (with 8 rows and no ring
  // whatever the storage, FP64 state, BF16, N=50000 took 0.802 ms against
  // 0.757 with 16 rows), and a run that comes to the dense form between
  // advances (from a factor, or with another storage), so that an evaluation
  // in between does not change the run.  Rows are summed in the same order in
  // every variant.  No HIP call when there is nothing to drop: safe under
  // capture.
  void ensure_variant() {
    if (!tuned && !factored && !sym()) default_variant();
  }

  int select_variant(int rows, int flags) override {
    if (rows != 4 && rows != 8 && rows != 16) return fail(KMT_ERR_ARG, "rows per group must be 4, 8 or 16 (got %d)", rows);
    if (flags & ~7) return fail(KMT_ERR_ARG, "unknown variant flags 0x%x", flags);
    if ((flags & 6) == 6) return fail(KMT_ERR_ARG, "the chunk ring has one workgroup per row group (not balanced)");
    tune_rows = rows;
    tune_nt = flags & 1;
    tune_bal = (flags >> 1) & 1;
    tune_ring = (flags >> 2) & 1;
    bal_grid = 0;
    tuned = pinned = 1;
    drop_graphs();
    return KMT_OK;
  }
  int tune(int reps, double *ms12) override {
    KMT_TRY(autotune(reps));
    if (ms12) for (int q = 0; q < 12; ++q) ms12[q] = tune_ms[q];
    return KMT_OK;
  }

  int set_omega(const void *om) override {
    HIP_TRY(hipMemcpyAsync(omega, om, sizeof(R) * N, hipMemcpyHostToDevice, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  int set_state(const void *th, double t, double h) override {
    HIP_TRY(hipMemcpyAsync(y, th, sizeof(R) * N, hipMemcpyHostToDevice, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    t0_ = (R)t;
    h0_ = (R)h;
    begun = 0;
    return KMT_OK;
  }

  int fetch_state() {
    if (fresh) return KMT_OK;
    HIP_TRY(hipMemcpyAsync(st_host, st, sizeof(State<R>), hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    shadow = *st_host;
    fresh = true;
    return KMT_OK;
  }

  int push_state() {
    *st_host = shadow;
    HIP_TRY(hipMemcpyAsync(st, st_host, sizeof(State<R>), hipMemcpyHostToDevice, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    fresh = true;
    dirty = false;
    return KMT_OK;
  }
  // before launches that change the state (fetch_state waits for them before
  // st_host is used again)
  int flush_state() {
    if (dirty) {
      *st_host = shadow;
      HIP_TRY(hipMemcpyAsync(st, st_host, sizeof(State<R>), hipMemcpyHostToDevice, stream));
      dirty = false;
    }
    fresh = false;
    return KMT_OK;
  }

  // `rows` rows of `width` bytes to the caller's memory.  What the runtime
  // knows (pinned, device or managed memory) is written by one copy.  A pitched
  // copy into pageable memory took 0.5 ms for six rows of 20 KB and 2 ms for
  // 190 of 40 KB; there whole stretches of the source go to a pinned half
  // buffer while the other half is spread over the caller's rows.  Without
  // pinned memory to be had, the pitched copy it is.
  int drain_rows(void *dst, const void *src, size_t pitch, size_t width, size_t rows) {
    hipPointerAttribute_t at{};
    const hipError_t known = hipPointerGetAttributes(&at, dst);
    if (known != hipSuccess) (void)hipGetLastError();  // an address the runtime does not know is no error here
    const bool direct = known == hipSuccess && at.type != hipMemoryTypeUnregistered;
    const size_t total = (rows - 1) * pitch + width;
    const size_t half = std::min(kStageMax, std::max<size_t>((total + 1) / 2, 4096));
    if (!direct && stage_half < half) {
      if (stage_buf) HIP_TRY(hipHostFree(stage_buf));
      stage_buf = nullptr;
      stage_half = 0;
      for (hipEvent_t &e : stage_ev)
        if (!e) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      if (hipHostMalloc((void **)&stage_buf, 2 * half, hipHostMallocDefault) == hipSuccess) {
        stage_half = half;
      } else {
        stage_buf = nullptr;
        (void)hipGetLastError();
      }
    }
    if (direct || !stage_buf) {
      HIP_TRY(hipMemcpy2DAsync(dst, width, src, pitch, width, rows, direct ? hipMemcpyDefault : hipMemcpyDeviceToHost, stream));
      return KMT_OK;
    }
    const size_t chunks = (total + stage_half - 1) / stage_half;
    auto start = [&](size_t c) -> int {
      const size_t o = c * stage_half, n = std::min(stage_half, total - o);
      HIP_TRY(hipMemcpyAsync(stage_buf + (c & 1) * stage_half, (const char *)src + o, n, hipMemcpyDeviceToHost, stream));
      HIP_TRY(hipEventRecord(stage_ev[c & 1], stream));
      return KMT_OK;
    };
    KMT_TRY(start(0));
    for (size_t c = 0; c < chunks; ++c) {
      if (c + 1 < chunks) KMT_TRY(start(c + 1));
      HIP_TRY(hipEventSynchronize(stage_ev[c & 1]));
      const size_t o = c * stage_half, end = o + std::min(stage_half, total - o);
      for (size_t q = o; q < end;) {  // the pieces of rows in [o, end)
        const size_t row = q / pitch, col = q % pitch, next = std::min(end, (row + 1) * pitch);
        if (col < width)
          std::memcpy((char *)dst + row * width + col, stage_buf + (c & 1) * stage_half + (q - o),
                      std::min(next - q, width - col));
        q = next;
      }
    }
    return KMT_OK;
  }

  int get_state(void *th, double *t, double *h) override {
    if (!begun) {
      HIP_TRY(hipMemcpyAsync(th, y, sizeof(R) * N, hipMemcpyDeviceToHost, stream));
      HIP_TRY(hipStreamSynchronize(stream));
      if (t) *t = (double)t0_;
      if (h) *h = (double)h0_;
      return KMT_OK;
    }
    KMT_TRY(fetch_state());
    const R *src = shadow.commit_pending ? ynew : y;
    HIP_TRY(hipMemcpyAsync(th, src, sizeof(R) * N, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    if (t) *t = (double)shadow.t;
    if (h) *h = (double)shadow.h;
    return KMT_OK;
  }

  // ---------------- adjacency ----------------
  size_t elem_bytes(int stg) const {
    const int el = stg & ~KMT_ADJ_SYM;
    return (el == KMT_ADJ_BF16 || el == KMT_ADJ_F16) ? 2 : sizeof(R);
  }
  static bool is_sym(int stg) { return stg >= 0 && (stg & KMT_ADJ_SYM); }
  bool sym() const { return is_sym(storage); }

  // block layout of KMT_ADJ_SYM: the (I, J) table and the partial buffers
  int ensure_sym() {
    if (sym_ij) return KMT_OK;
    sym_nb = (N + kSymT - 1) / kSymT;
    sym_blocks = sym_nb * (sym_nb + 1) / 2;
    std::vector<int2> ij((size_t)sym_blocks);
    for (long I = 0; I < sym_nb; ++I)
      for (long J = I; J < sym_nb; ++J) ij[(size_t)sym_index(I, J, sym_nb)] = make_int2((int)I, (int)J);
    HIP_TRY(hipMalloc((void **)&sym_ij, sizeof(int2) * ij.size()));
    HIP_TRY(hipMemcpyAsync(sym_ij, ij.data(), sizeof(int2) * ij.size(), hipMemcpyHostToDevice, stream));
    // sized for the wider of the accumulation types (double for native
    // storage, float for 16-bit storage)
    HIP_TRY(hipMalloc((void **)&sym_prow, sizeof(SymPair<double>) * (size_t)sym_blocks * kSymT));
    HIP_TRY(hipMalloc((void **)&sym_pcol, sizeof(SymPair<double>) * (size_t)sym_blocks * kSymT));
    HIP_TRY(hipMemsetAsync(sym_prow, 0, sizeof(SymPair<double>) * (size_t)sym_blocks * kSymT, stream));
    HIP_TRY(hipMemsetAsync(sym_pcol, 0, sizeof(SymPair<double>) * (size_t)sym_blocks * kSymT, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  int ensure_A(int stg) {
    const int el = stg & ~KMT_ADJ_SYM;
    if (stg < 0 || (el != KMT_ADJ_NATIVE && el != KMT_ADJ_BF16 && el != KMT_ADJ_F16))
      return fail(KMT_ERR_ARG, "unknown adjacency storage %d", stg);
    if (is_sym(stg)) {
      KMT_TRY(ensure_sym());
    } else if (sym_ij) {  // back to row-major storage: drop the block table and partials
      drop_graphs();
      HIP_TRY(hipStreamSynchronize(stream));
      (void)hipFree(sym_ij);
      (void)hipFree(sym_prow);
      (void)hipFree(sym_pcol);
      sym_ij = nullptr;
      sym_prow = sym_pcol = nullptr;
    }
    const size_t bytes = is_sym(stg) ? (size_t)sym_blocks * kSymT * kSymT * elem_bytes(stg)
                                     : (size_t)rows_alloc * (size_t)lda * elem_bytes(stg);
    if (A && A_bytes == bytes && storage == stg) return KMT_OK;
    drop_graphs();
    if (A) {
      HIP_TRY(hipStreamSynchronize(stream));
      HIP_TRY(hipFree(A));
      A = nullptr;
    }
    hipError_t e = hipMalloc(&A, bytes);
    if (e != hipSuccess) {
      A = nullptr;
      return fail(KMT_ERR_MEMORY, "cannot allocate %zu bytes for the adjacency: %s", bytes, hipGetErrorString(e));
    }
    A_bytes = bytes;
    storage = stg;
    tuned = pinned = 0;
    bal_grid = 0;
    HIP_TRY(hipMemsetAsync(A, 0, bytes, stream));
    return KMT_OK;
  }

  static double pow2_at_least(double v) {
    if (!(v > 0) || !std::isfinite(v)) return 1.0;
    return std::ldexp(1.0, (int)std::ceil(std::log2(v)));
  }

  template <class S> int upload_rows(const R *M, long ld, R inv_scale) {
    // stage rows through a device buffer, convert into the stored layout
    const long chunk = std::max<long>(1, std::min<long>(N, (64l << 20) / (long)(sizeof(R) * N)));
    R *stage = nullptr;
    HIP_TRY(hipMalloc((void **)&stage, sizeof(R) * chunk * N));
    for (long r0 = 0; r0 < N; r0 += chunk) {
      const long nr = std::min(chunk, N - r0);
      hipError_t e = hipMemcpy2DAsync(stage, sizeof(R) * N, M + (size_t)r0 * ld, sizeof(R) * ld, sizeof(R) * N, nr,
                                      hipMemcpyHostToDevice, stream);
      if (e == hipSuccess) {
        dim3 grid((unsigned)std::min<long>((N + kBlock - 1) / kBlock, 64), (unsigned)nr);
        convert_rows_kernel<R, S><<<grid, kBlock, 0, stream>>>(stage, N, N, nr, (S *)A + (size_t)r0 * lda, lda, inv_scale);
        e = hipGetLastError();
      }
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
      if (e != hipSuccess) {
        (void)hipFree(stage);
        return fail(KMT_ERR_HIP, "adjacency upload failed: %s", hipGetErrorString(e));
      }
    }
    HIP_TRY(hipFree(stage));
    return KMT_OK;
  }

  int set_adjacency(const void *Mv, int src_prec, long ld, int stg) override {
    if (ld < N) return fail(KMT_ERR_ARG, "adjacency row stride %ld < N=%ld", ld, N);
    HIP_TRY(hipStreamSynchronize(stream));
    drop_graphs();  // captured launches hold the old matrix scale
    if (src_prec != (sizeof(R) == 4 ? KMT_F32 : KMT_F64))
      return fail(KMT_ERR_ARG, "adjacency source precision must match the context precision");
    const R *M = (const R *)Mv;
    if (is_sym(stg)) {
      for (long i = 0; i < N; ++i)
        for (long j = i + 1; j < N; ++j)
          if (!(M[(size_t)i * ld + j] == M[(size_t)j * ld + i]) &&
              !(std::isnan((double)M[(size_t)i * ld + j]) && std::isnan((double)M[(size_t)j * ld + i])))
            return fail(KMT_ERR_ARG, "KMT_ADJ_SYM needs a symmetric matrix: M[%ld][%ld] != M[%ld][%ld]", i, j, j, i);
      KMT_TRY(ensure_A(stg));
      factored = 0;
      mscale_ = 1.0;
      if ((stg & ~KMT_ADJ_SYM) == KMT_ADJ_NATIVE) return upload_sym<R>(M, ld, (R)1);
      double mx = 0;
      for (long i = 0; i < N; ++i)
        for (long j = 0; j < N; ++j) mx = std::max(mx, std::fabs((double)M[(size_t)i * ld + j]));
      mscale_ = pow2_at_least(mx);
      const R inv = (R)(1.0 / mscale_);
      if ((stg & ~KMT_ADJ_SYM) == KMT_ADJ_BF16) return upload_sym<bf16_t>(M, ld, inv);
      return upload_sym<f16_t>(M, ld, inv);
    }
    KMT_TRY(ensure_A(stg));
    if (stg == KMT_ADJ_NATIVE) {
      mscale_ = 1.0;
      HIP_TRY(hipMemcpy2DAsync(A, sizeof(R) * lda, M, sizeof(R) * ld, sizeof(R) * N, N, hipMemcpyHostToDevice, stream));
      HIP_TRY(hipStreamSynchronize(stream));
      factored = 0;
      return KMT_OK;
    }
    double mx = 0;
    for (long i = 0; i < N; ++i)
      for (long j = 0; j < N; ++j) mx = std::max(mx, std::fabs((double)M[(size_t)i * ld + j]));
    mscale_ = pow2_at_least(mx);
    factored = 0;
    const R inv = (R)(1.0 / mscale_);
    if (stg == KMT_ADJ_BF16) return upload_rows<bf16_t>(M, ld, inv);
    return upload_rows<f16_t>(M, ld, inv);
  }

  // pack the upper block triangle of a host matrix, a few blocks per copy,
  // through a device staging buffer converted into the stored type
  template <class S> int upload_sym(const R *M, long ld, R inv_scale) {
    const long per = 32;
    std::vector<R> buf((size_t)per * kSymT * kSymT);
    R *stage = nullptr;
    HIP_TRY(hipMalloc((void **)&stage, sizeof(R) * buf.size()));
    for (long b0 = 0; b0 < sym_blocks; b0 += per) {
      const long nbk = std::min(per, sym_blocks - b0);
      std::fill(buf.begin(), buf.end(), (R)0);
      long b = 0;
      for (long I = 0; I < sym_nb && b < b0 + nbk; ++I)
        for (long J = I; J < sym_nb; ++J, ++b) {
          if (b < b0) continue;
          if (b >= b0 + nbk) break;
          R *dst = buf.data() + (size_t)(b - b0) * kSymT * kSymT;
          for (long r = 0; r < kSymT && I * kSymT + r < N; ++r)
            for (long c = 0; c < kSymT && J * kSymT + c < N; ++c)
              dst[(size_t)r * kSymT + c] = M[(size_t)(I * kSymT + r) * ld + J * kSymT + c];
        }
      hipError_t e = hipMemcpyAsync(stage, buf.data(), sizeof(R) * (size_t)nbk * kSymT * kSymT, hipMemcpyHostToDevice,
                                    stream);
      if (e == hipSuccess) {
        dim3 grid(1, (unsigned)(nbk * kSymT));
        convert_rows_kernel<R, S><<<grid, kBlock, 0, stream>>>(stage, kSymT, kSymT, nbk * kSymT,
                                                               (S *)A + (size_t)b0 * kSymT * kSymT, kSymT, inv_scale);
        e = hipGetLastError();
      }
      if (e == hipSuccess) e = hipStreamSynchronize(stream);  // buf is refilled next
      if (e != hipSuccess) {
        (void)hipFree(stage);
        return fail(KMT_ERR_HIP, "adjacency upload failed: %s", hipGetErrorString(e));
      }
    }
    HIP_TRY(hipFree(stage));
    return KMT_OK;
  }

  int set_factor(const void *Xv, const void *wv, int k_) override {
    if (k_ < 0) return fail(KMT_ERR_ARG, "rank K must be >= 0");
    HIP_TRY(hipStreamSynchronize(stream));  // the buffers below may be in use by queued work
    drop_graphs();
    drop_factor();
    const int rc = make_factor(Xv, wv, k_);
    if (rc != KMT_OK) {  // all of it or none: coupling_ready asks for X alone
      drop_factor();
      return rc;
    }
    if (factored == KMT_LOWRANK_REBUILD) {  // keep the mode, if the new rank allows it
      factored = KMT_LOWRANK_CONTRACT;
      return use_factored(KMT_LOWRANK_REBUILD);
    }
    return KMT_OK;
  }

  void drop_factor() {
    if (X) { (void)hipFree(X); X = nullptr; }
    if (w) { (void)hipFree(w); w = nullptr; }
    if (XT) { (void)hipFree(XT); XT = nullptr; }
    if (lr_part) { (void)hipFree(lr_part); lr_part = nullptr; }
    if (lr_G) { (void)hipFree(lr_G); lr_G = nullptr; }
    drop_sign();
  }

  int make_factor(const void *Xv, const void *wv, int k_) {
    K = k_;
    const long kk = std::max(K, 1);
    X_host.assign((const R *)Xv, (const R *)Xv + (size_t)N * K);
    w_host.assign((const R *)wv, (const R *)wv + K);
    HIP_TRY(hipMalloc((void **)&X, sizeof(R) * std::max<size_t>((size_t)N * K, 1)));
    HIP_TRY(hipMalloc((void **)&w, sizeof(R) * kk));
    if (K > 0) {
      HIP_TRY(hipMemcpyAsync(X, Xv, sizeof(R) * N * K, hipMemcpyHostToDevice, stream));
      HIP_TRY(hipMemcpyAsync(w, wv, sizeof(R) * K, hipMemcpyHostToDevice, stream));
    }
    lr_nblk = (int)std::min<long>((N + kBlock - 1) / kBlock, 512);
    lr_blocks = (int)std::min<long>((N + kBlock - 1) / kBlock, kLrMaxBlocks);
    const int nparts = std::max(lr_nblk, 3 * lr_blocks);
    if (K <= kLrMaxRank) {
      KMT_TRY(alloc_vec(&XT, (long)kk * ldv));
      transpose_factor_kernel<R><<<(unsigned)((N + kBlock - 1) / kBlock), kBlock, 0, stream>>>(X, K, N, ldv, XT);
      HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipMalloc((void **)&lr_part, sizeof(double) * 2 * kk * nparts));
    HIP_TRY(hipMemsetAsync(lr_part, 0, sizeof(double) * 2 * kk * nparts, stream));
    HIP_TRY(hipMalloc((void **)&lr_G, sizeof(double) * 2 * kk));
    HIP_TRY(hipMemsetAsync(lr_G, 0, sizeof(double) * 2 * kk, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  void drop_sign() {
    void *b[] = {s_pass[0].tiles, s_pass[0].bfrag, s_pass[0].ones, s_pass[1].tiles, s_pass[1].bfrag, s_pass[1].ones};
    for (void *p : b)
      if (p) (void)hipFree(p);
    s_pass[0] = s_pass[1] = SignPass();
    sign = 0;
  }

  // 16-row tiles per wave of the int8 passes
  static constexpr int kSignNT = 4;
  // Shape of a pass with `rows` output rows (+ the ones row) over kdim: the
  // (row group, pair) units in equal stretches over the workgroups that the
  // device holds at once, at least 2 pairs each (a pass of N = K = 10^4 is
  // 400 units, 200 workgroups: latency-bound either way, and fewer partials).
  static constexpr long kSignRowsPerBlock = 16 * kSignNT * (kBlock / kWave);
  static SignPass sign_pass_shape(long rows, long kdim, long resident) {
    SignPass p;
    p.ldp = (rows + 1 + kSignRowsPerBlock - 1) / kSignRowsPerBlock * kSignRowsPerBlock;
    const long groups = p.ldp / kSignRowsPerBlock;
    p.npairs = std::max<long>(1, (kdim + 2 * kSignSB - 1) / (2 * kSignSB));
    p.nsb = 2 * p.npairs;
    p.units = groups * p.npairs;
    p.wgs = (int)std::min(resident, std::max<long>(1, p.units / 2));
    p.nsplit = 1;
    for (long g = 0; g < groups; ++g)
      p.nsplit = std::max(p.nsplit, (int)(sign_unit_owner((g + 1) * p.npairs - 1, p.units, p.wgs) -
                                          sign_unit_owner(g * p.npairs, p.units, p.wgs) + 1));
    return p;
  }
  int alloc_sign_pass(SignPass &p, long kdim) {
    // one allocation, cleared once: columns past the vectors' end and slots
    // that a row group does not reach stay zero
    const size_t frag_bytes = (size_t)p.nsb * 8 * kWave * 16, nfrag = &p == &s_pass[0] ? 2 : 1;
    const size_t part_bytes = sizeof(int32_t) * 16 * (size_t)p.nsplit * p.ldp;
    HIP_TRY(hipMalloc((void **)&p.bfrag, nfrag * frag_bytes + part_bytes));
    HIP_TRY(hipMemsetAsync(p.bfrag, 0, nfrag * frag_bytes + part_bytes, stream));
    if (nfrag == 2) p.bfrag_rhs = p.bfrag + frag_bytes;
    p.part = (int32_t *)(p.bfrag + nfrag * frag_bytes);
    std::vector<uint32_t> ones((size_t)16 * p.nsb, 0u);
    for (long q = 0; q < (long)ones.size(); ++q)
      ones[q] = 32 * (q + 1) <= kdim ? 0xFFFFFFFFu : (32 * q < kdim ? (1u << (kdim - 32 * q)) - 1u : 0u);
    HIP_TRY(hipMalloc((void **)&p.ones, sizeof(uint32_t) * ones.size()));
    HIP_TRY(hipMemcpy(p.ones, ones.data(), sizeof(uint32_t) * ones.size(), hipMemcpyHostToDevice));
    return KMT_OK;
  }

  // The volcano factor X_nm = +-1 of the library's sign stream, packed, and
  // w_m = (-1)^m / N (makeu1 / makeu2 / m1 / m2, kuramoto.cu:62-143).
  int set_factor_sign(int k_, uint32_t seed) override {
    if (k_ < 0) return fail(KMT_ERR_ARG, "rank K must be >= 0");
    if (N > kSignMaxDim || k_ > kSignMaxDim)
      return fail(KMT_ERR_ARG, "the packed sign factor needs N, K <= %ld (N=%ld, K=%d)", kSignMaxDim, N, k_);
    HIP_TRY(hipStreamSynchronize(stream));
    drop_graphs();
    drop_factor();
    if (factored == KMT_LOWRANK_REBUILD) factored = KMT_LOWRANK_CONTRACT;
    K = k_;
    X_host.clear();
    w_host.assign((size_t)K, (R)0);
    for (int m = 0; m < K; ++m) w_host[m] = (R)(((m & 1) ? -1.0 : 1.0) / (double)N);
    HIP_TRY(hipMalloc((void **)&w, sizeof(R) * std::max(K, 1)));
    if (K > 0) HIP_TRY(hipMemcpyAsync(w, w_host.data(), sizeof(R) * K, hipMemcpyHostToDevice, stream));
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, sign_mfma_kernel<R, kSignNT>, kBlock, 0) != hipSuccess ||
        per_cu < 1)
      per_cu = 1;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1) cus = 1;
    const long resident = (long)per_cu * cus;
    s_pass[0] = sign_pass_shape(K, N, resident);
    s_pass[1] = sign_pass_shape(N, K, resident);
    SignPass &p1 = s_pass[0], &p2 = s_pass[1];
    const size_t tw1 = (size_t)p1.ldp * 32 * p1.npairs, tw2 = (size_t)p2.ldp * 32 * p2.npairs;
    hipError_t e = hipMalloc((void **)&p1.tiles, sizeof(uint32_t) * tw1);
    if (e == hipSuccess) e = hipMalloc((void **)&p2.tiles, sizeof(uint32_t) * tw2);
    if (e != hipSuccess) {
      drop_sign();
      return fail(KMT_ERR_MEMORY, "cannot allocate the packed sign factor (N=%ld, K=%d): %s", N, K, hipGetErrorString(e));
    }
    if (alloc_sign_pass(p1, N) != KMT_OK || alloc_sign_pass(p2, K) != KMT_OK) {
      drop_sign();
      return fail(KMT_ERR_MEMORY, "cannot allocate the sign passes' buffers (N=%ld, K=%d)", N, K);
    }
    // zero rows (and words past each row's k range) stay as cleared here
    HIP_TRY(hipMemsetAsync(p1.tiles, 0, sizeof(uint32_t) * tw1, stream));
    HIP_TRY(hipMemsetAsync(p2.tiles, 0, sizeof(uint32_t) * tw2, stream));
    const size_t words = (size_t)((N + 255) / 256) * p2.npairs * 8192;
    gen_sign_bits_kernel<<<(unsigned)((words + kBlock - 1) / kBlock), kBlock, 0, stream>>>(p2.tiles, N, K, p2.npairs,
                                                                                          seed);
    HIP_TRY(hipGetLastError());
    if (K > 0) {
      const long kw = (K + 31) / 32;
      const size_t waves = (size_t)((N + 63) / 64) * kw;
      transpose_sign_bits_kernel<<<(unsigned)((waves * kWave + kBlock - 1) / kBlock), kBlock, 0, stream>>>(
          p2.tiles, N, p2.npairs, kw, p1.tiles, p1.npairs);
      HIP_TRY(hipGetLastError());
    }
    // the ones rows last: the transpose writes zero words into rows m >= K
    sign_tile_ones_kernel<<<(unsigned)((32 * p1.npairs + kBlock - 1) / kBlock), kBlock, 0, stream>>>(
        p1.tiles, K, p1.ones, p1.npairs);
    sign_tile_ones_kernel<<<(unsigned)((32 * p2.npairs + kBlock - 1) / kBlock), kBlock, 0, stream>>>(
        p2.tiles, N, p2.ones, p2.npairs);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(stream));
    sign = 1;
    return KMT_OK;
  }

  template <class S> int gen_sign_rows(R inv_scale) {
    constexpr int ROWS = 8;
    const long chunk = 4096;
    for (long r0 = 0; r0 < N; r0 += chunk) {
      const long nr = std::min(chunk, N - r0);
      dim3 grid((unsigned)((N + kBlock - 1) / kBlock), (unsigned)((nr + ROWS - 1) / ROWS));
      gen_adj_sign_kernel<R, S, ROWS><<<grid, kBlock, 0, stream>>>(s_pass[1].tiles, s_pass[1].npairs, w, K, N, r0, nr,
                                                                   (S *)A + (size_t)r0 * lda, lda, inv_scale);
      HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  template <class S> int gen_rows(R inv_scale) {
    const long chunk = 4096;
    for (long r0 = 0; r0 < N; r0 += chunk) {
      const long nr = std::min(chunk, N - r0);
      gen_adj_kernel<R, S><<<(unsigned)nr, kBlock, 0, stream>>>(X, w, K, N, r0, (S *)A + (size_t)r0 * lda, lda, inv_scale);
      HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  int build_adjacency(int stg) override {
    if (!X && !sign) return fail(KMT_ERR_STATE, "kmt_build_adjacency needs kmt_set_factor or kmt_set_factor_sign first");
    if (sign && is_sym(stg)) return fail(KMT_ERR_ARG, "symmetric storage is not built from a packed sign factor");
    HIP_TRY(hipStreamSynchronize(stream));
    drop_graphs();  // captured launches hold the old matrix scale
    KMT_TRY(ensure_A(stg));
    factored = 0;
    if (sign) {
      // |M_ij| <= sum_m |w_m| (X^2 = 1): scale the 16-bit forms so |stored| <= 1
      double mx = 0;
      for (int m = 0; m < K; ++m) mx += std::fabs((double)w_host[m]);
      mscale_ = stg == KMT_ADJ_NATIVE ? 1.0 : pow2_at_least(mx);
      const R inv = (R)(1.0 / mscale_);
      if (stg == KMT_ADJ_NATIVE) return gen_sign_rows<R>((R)1);
      if (stg == KMT_ADJ_BF16) return gen_sign_rows<bf16_t>(inv);
      return gen_sign_rows<f16_t>(inv);
    }
    if (stg == KMT_ADJ_NATIVE) {
      mscale_ = 1.0;
      return gen_rows<R>((R)1);
    }
    if (stg == KMT_ADJ_SYM) {
      mscale_ = 1.0;
      gen_adj_sym_kernel<R, R><<<(unsigned)sym_blocks, kBlock, 0, stream>>>(X, w, K, N, sym_ij, (R *)A, (R)1);
      HIP_TRY(hipGetLastError());
      HIP_TRY(hipStreamSynchronize(stream));
      return KMT_OK;
    }
    // |M_ij| <= max_n sum_m |w_m| X_nm^2 (Cauchy–Schwarz): scale so |stored| <= 1
    double mx = 0;
    for (long n = 0; n < N; ++n) {
      double s = 0;
      for (int m = 0; m < K; ++m) s += std::fabs((double)w_host[m]) * (double)X_host[n * K + m] * (double)X_host[n * K + m];
      mx = std::max(mx, s);
    }
    mscale_ = pow2_at_least(mx);
    const R inv = (R)(1.0 / mscale_);
    if (is_sym(stg)) {
      if ((stg & ~KMT_ADJ_SYM) == KMT_ADJ_BF16)
        gen_adj_sym_kernel<R, bf16_t><<<(unsigned)sym_blocks, kBlock, 0, stream>>>(X, w, K, N, sym_ij, (bf16_t *)A, inv);
      else
        gen_adj_sym_kernel<R, f16_t><<<(unsigned)sym_blocks, kBlock, 0, stream>>>(X, w, K, N, sym_ij, (f16_t *)A, inv);
      HIP_TRY(hipGetLastError());
      HIP_TRY(hipStreamSynchronize(stream));
      return KMT_OK;
    }
    if (stg == KMT_ADJ_BF16) return gen_rows<bf16_t>(inv);
    return gen_rows<f16_t>(inv);
  }

  int use_factored(int on) override {
    if (on < 0 || on > KMT_LOWRANK_REBUILD) return fail(KMT_ERR_ARG, "unknown low-rank mode %d", on);
    if (on && !X && !sign) return fail(KMT_ERR_STATE, "-A needs kmt_set_factor or kmt_set_factor_sign first");
    if (on == KMT_LOWRANK_REBUILD && sign)
      return fail(KMT_ERR_ARG, "register-rebuilt tiles need a real factor (kmt_set_factor), not a packed sign factor");
    if (on == KMT_LOWRANK_REBUILD && K > kLrMaxRank)
      return fail(KMT_ERR_ARG, "register-rebuilt tiles support K <= %d (K=%d)", kLrMaxRank, K);
    if (factored != on) drop_graphs();
    factored = on;
    return KMT_OK;
  }

  int get_adjacency_rows(long i0, long i1, void *out) override {
    if (!A) return fail(KMT_ERR_STATE, "no dense adjacency on the device");
    if (i0 < 0 || i1 > N || i0 > i1) return fail(KMT_ERR_ARG, "row range [%ld, %ld) outside [0, %ld)", i0, i1, N);
    const long chunk = std::max<long>(1, std::min<long>(i1 - i0, (64l << 20) / (long)(sizeof(R) * N)));
    R *stage = nullptr;
    HIP_TRY(hipMalloc((void **)&stage, sizeof(R) * chunk * N));
    for (long r0 = i0; r0 < i1; r0 += chunk) {
      const long nr = std::min(chunk, i1 - r0);
      dim3 grid((unsigned)std::min<long>((N + kBlock - 1) / kBlock, 64), (unsigned)nr);
      hipError_t e = hipSuccess;
      if (storage == KMT_ADJ_SYM)
        read_sym_rows_kernel<R, R><<<grid, kBlock, 0, stream>>>((const R *)A, sym_nb, N, r0, nr, (R)1, stage);
      else if (storage == (KMT_ADJ_SYM | KMT_ADJ_BF16))
        read_sym_rows_kernel<R, bf16_t><<<grid, kBlock, 0, stream>>>((const bf16_t *)A, sym_nb, N, r0, nr, (R)mscale_, stage);
      else if (storage == (KMT_ADJ_SYM | KMT_ADJ_F16))
        read_sym_rows_kernel<R, f16_t><<<grid, kBlock, 0, stream>>>((const f16_t *)A, sym_nb, N, r0, nr, (R)mscale_, stage);
      else if (storage == KMT_ADJ_NATIVE)
        read_rows_kernel<R, R><<<grid, kBlock, 0, stream>>>((const R *)A + (size_t)r0 * lda, lda, N, nr, (R)1, stage);
      else if (storage == KMT_ADJ_BF16)
        read_rows_kernel<R, bf16_t><<<grid, kBlock, 0, stream>>>((const bf16_t *)A + (size_t)r0 * lda, lda, N, nr, (R)mscale_, stage);
      else
        read_rows_kernel<R, f16_t><<<grid, kBlock, 0, stream>>>((const f16_t *)A + (size_t)r0 * lda, lda, N, nr, (R)mscale_, stage);
      e = hipGetLastError();
      if (e == hipSuccess) e = hipMemcpyAsync((R *)out + (size_t)(r0 - i0) * N, stage, sizeof(R) * nr * N, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
      if (e != hipSuccess) {
        (void)hipFree(stage);
        return fail(KMT_ERR_HIP, "adjacency read failed: %s", hipGetErrorString(e));
      }
    }
    HIP_TRY(hipFree(stage));
    return KMT_OK;
  }

  // ---------------- launches ----------------
  Vecs<R> vecs(const R *cs_in, R *cs_out, int check) {
    Vecs<R> v;
    v.cs_in = cs_in;
    v.cs_out = cs_out;
    v.ldv = ldv;
    v.N = N;
    v.omega = omega;
    v.y = y;
    for (int j = 0; j < 7; ++j) v.k[j] = k[j];
    v.ynew = ynew;
    v.f_out = f_scr;
    v.cs_pairs = nullptr;
    v.c1 = c1;
    v.st = st;
    v.err_part = err_part;
    v.check_state = check;
    return v;
  }

  int coupling_ready() const { return factored ? (X != nullptr || sign) : (A != nullptr); }
  // before attempts are launched: kmt_use_factored and failed uploads can take
  // the coupling away from a run between advances
  int still_coupled() const {
    if (!coupling_ready()) return fail(KMT_ERR_STATE, "no adjacency: call kmt_set_adjacency, kmt_build_adjacency or kmt_set_factor + kmt_use_factored");
    return KMT_OK;
  }

  // workgroups of one resident round of the balanced variant (<= N rows)
  template <class S, int ROWS, bool NT> int balanced_grid() {
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, stage_kernel<R, S, ROWS, 3, NT, true>, kBlock, 0) !=
            hipSuccess || per_cu < 1)
      per_cu = 1;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1) cus = 1;
    return (int)std::min<long>(std::min<long>((long)per_cu * cus, N), n_err_part);
  }

  template <class S, int KIND, int ROWS, bool NT> void launch_dense_variant(const DenseArgs<R, S> &a) {
    if (tune_bal) {
      if (bal_grid <= 0) bal_grid = balanced_grid<S, ROWS, NT>();
      stage_kernel<R, S, ROWS, KIND, NT, true><<<(unsigned)bal_grid, kBlock, 0, stream>>>(a);
    } else if (tune_ring && (pinned || ROWS < 16 || sizeof(S) > 2)) {
      const unsigned grid = (unsigned)((N + ROWS - 1) / ROWS);
      stage_ring_kernel<R, S, ROWS, KIND, NT><<<grid, kBlock, 0, stream>>>(a);
    } else {
      const unsigned grid = (unsigned)((N + ROWS - 1) / ROWS);
      stage_kernel<R, S, ROWS, KIND, NT, false><<<grid, kBlock, 0, stream>>>(a);
    }
  }

  template <class S, int KIND> void launch_dense_kind(const Vecs<R> &v) {
    DenseArgs<R, S> a;
    a.A = (const S *)A;
    a.lda = lda;
    a.mscale = (R)mscale_;
    a.v = v;
    switch ((KIND == 7 ? error_rows() : tune_rows) * 2 + (tune_nt ? 1 : 0)) {
      case 8: launch_dense_variant<S, KIND, 4, false>(a); break;
      case 9: launch_dense_variant<S, KIND, 4, true>(a); break;
      case 16: launch_dense_variant<S, KIND, 8, false>(a); break;
      case 32: launch_dense_variant<S, KIND, 16, false>(a); break;
      case 33: launch_dense_variant<S, KIND, 16, true>(a); break;
      default: launch_dense_variant<S, KIND, 8, true>(a); break;
    }
  }

  // KMT_ADJ_SYM: block kernel over the stored triangle, then the row reduction
  template <class S, int KIND> void launch_sym_as(const Vecs<R> &v) {
    using Acc = typename Store<S>::Acc;
    SymArgs<R, S> a;
    a.A = (const S *)A;
    a.ij = sym_ij;
    a.nb = sym_nb;
    a.prow = reinterpret_cast<SymPair<Acc> *>(sym_prow);
    a.pcol = reinterpret_cast<SymPair<Acc> *>(sym_pcol);
    a.mscale = (R)mscale_;
    a.v = v;
    sym_tile_kernel<R, S><<<(unsigned)sym_blocks, kBlock, 0, stream>>>(a);
    sym_reduce_kernel<R, S, KIND><<<(unsigned)sym_nb, kBlock, 0, stream>>>(a);
  }
  template <int KIND> void launch_sym(const Vecs<R> &v) {
    if (storage == KMT_ADJ_SYM) launch_sym_as<R, KIND>(v);
    else if (storage == (KMT_ADJ_SYM | KMT_ADJ_BF16)) launch_sym_as<bf16_t, KIND>(v);
    else launch_sym_as<f16_t, KIND>(v);
  }

  template <int KIND> void launch_dense(const Vecs<R> &v) {
    if (sym()) launch_sym<KIND>(v);
    else if (storage == KMT_ADJ_NATIVE) launch_dense_kind<R, KIND>(v);
    else if (storage == KMT_ADJ_BF16) launch_dense_kind<bf16_t, KIND>(v);
    else launch_dense_kind<f16_t, KIND>(v);
  }

  bool lr_fused() const { return K <= kLrMaxRank && !sign; }
  bool lr_path() const { return factored == KMT_LOWRANK_CONTRACT && lr_fused(); }
  // partial-sum buffers of the fused low-rank path: 0 and 1 alternate between
  // the stages of an attempt (0: also the stage-2 vector's, kept between
  // attempts), 2 belongs to stand-alone right-hand sides
  double *lr_p(int which) const { return lr_part + (size_t)which * 2 * std::max(K, 1) * lr_blocks; }
  LrArgs<R> lr_args(int pin, int pout) const {
    LrArgs<R> l;
    l.XT = XT;
    l.w = w;
    l.K = K;
    l.blocks = lr_blocks;
    l.part_in = lr_p(pin);
    l.part_out = lr_p(pout);
    return l;
  }
  // the launch: one block per workgroup, or two
  int lr_threads() const { return lr_blocks > kLrPairedBlocks ? kLrThreads : kBlock; }
  unsigned lr_grid() const { return (unsigned)(lr_blocks > kLrPairedBlocks ? (lr_blocks + 1) / 2 : lr_blocks); }
  // f(rank bound, exact) for this context's rank
  template <class F> void lr_dispatch(F &&f) {
    using std::integral_constant;
    switch (K) {
      case 0: f(integral_constant<int, 1>{}, std::false_type{}); break;
      case 1: f(integral_constant<int, 1>{}, std::true_type{}); break;
      case 2: f(integral_constant<int, 2>{}, std::true_type{}); break;
      case 3: f(integral_constant<int, 3>{}, std::true_type{}); break;
      case 4: f(integral_constant<int, 4>{}, std::true_type{}); break;
      case 5: f(integral_constant<int, 5>{}, std::true_type{}); break;
      case 6: f(integral_constant<int, 6>{}, std::true_type{}); break;
      case 7: f(integral_constant<int, 7>{}, std::true_type{}); break;
      case 8: f(integral_constant<int, 8>{}, std::true_type{}); break;
      default: f(integral_constant<int, kLrMaxRank>{}, std::false_type{}); break;
    }
  }
  void launch_gram(const R *cs_in, int pout) {
    lr_dispatch([&](auto kt, auto exact) {
      lowrank_gram_kernel<R, decltype(kt)::value, decltype(exact)::value>
          <<<lr_grid(), lr_threads(), 0, stream>>>(lr_args(0, pout), N, cs_in, ldv);
    });
  }
  // stage KIND from the partials in lr_p(pin); stages 2..6 write those of
  // their output vector into lr_p(pout)
  template <int KIND> void launch_lr_stage(const Vecs<R> &v, int pin, int pout) {
    lr_dispatch([&](auto kt, auto exact) {
      lowrank_stage_kernel<R, KIND, decltype(kt)::value, decltype(exact)::value>
          <<<lr_grid(), lr_threads(), 0, stream>>>(lr_args(pin, pout), v);
    });
  }
  // one attempt's six stages on the fused low-rank path, one launch each
  // (the stage-2 vector's partials: the previous emit)
  void launch_lr_attempt(std::vector<std::pair<hipEvent_t, hipEvent_t>> *ev) {
    for (int s = 2; s <= 7; ++s) {
      const R *in = cs[(s - 2) & 1];
      R *out = cs[(s - 1) & 1];
      Vecs<R> v = vecs(in, out, 1);
      const int pin = (s - 2) & 1;
      if (ev) (void)hipEventRecord((*ev)[0].first, stream);
      switch (s) {
        case 2: launch_lr_stage<2>(v, pin, pin ^ 1); break;
        case 3: launch_lr_stage<3>(v, pin, pin ^ 1); break;
        case 4: launch_lr_stage<4>(v, pin, pin ^ 1); break;
        case 5: launch_lr_stage<5>(v, pin, pin ^ 1); break;
        case 6: launch_lr_stage<6>(v, pin, pin ^ 1); break;
        default: launch_lr_stage<7>(v, pin, pin ^ 1); break;
      }
      if (ev) {
        (void)hipEventRecord((*ev)[0].second, stream);
        ev->erase(ev->begin());
      }
    }
  }

  bool sign_path() const { return factored && sign; }
  unsigned vec_blocks(long n) const { return (unsigned)((n + kBlock - 1) / kBlock); }
  void launch_sign_limbs(const R *cs_in, uint8_t *bfrag) {
    if (K > 0) sign_limbs_kernel<R><<<vec_blocks(N), kBlock, 0, stream>>>(cs_in, cs_in + ldv, N, bfrag);
  }
  // packed sign factor: pass 1 (rows m) over the vector's digits, G as digits,
  // pass 2 (rows n), sums + stage epilogue.  An attempt's stages find their
  // vector's digits in the pass's own buffer (from the launch that wrote the
  // vector); a stand-alone right-hand side makes them in its own.
  template <int KIND> void launch_sign(const Vecs<R> &v) {
    const bool attempt = v.check_state && KIND >= 2;
    const int chk = attempt;
    const SignPass &p1 = s_pass[0], &p2 = s_pass[1];
    if (K > 0) {
      uint8_t *vec = attempt ? p1.bfrag : p1.bfrag_rhs;
      if (!attempt) launch_sign_limbs(v.cs_in, vec);
      sign_mfma_kernel<R, kSignNT><<<(unsigned)p1.wgs, kBlock, 0, stream>>>(
          (const u32x4 *)p1.tiles, (const u32x4 *)vec, (int)p1.npairs, p1.units, p1.part, p1.ldp, st, chk);
      sign_gram_kernel<R><<<vec_blocks(K), kBlock, 0, stream>>>(p1.part, p1.nsplit, p1.ldp, w, K, p2.bfrag, st, chk);
      sign_mfma_kernel<R, kSignNT><<<(unsigned)p2.wgs, kBlock, 0, stream>>>(
          (const u32x4 *)p2.tiles, (const u32x4 *)p2.bfrag, (int)p2.npairs, p2.units, p2.part, p2.ldp, st, chk);
    }
    sign_stage_kernel<R, KIND><<<vec_blocks(N), kBlock, 0, stream>>>(p2.part, K > 0 ? p2.nsplit : 0, p2.ldp, v,
                                                                     attempt && K > 0 ? p1.bfrag : nullptr);
  }

  template <int KIND> void launch_factored(const Vecs<R> &v) {
    if (sign) {
      launch_sign<KIND>(v);
      return;
    }
    if (lr_fused()) {
      launch_gram(v.cs_in, 2);
      launch_lr_stage<KIND>(v, 2, 1);
      return;
    }
    const int tiles = std::max(1, (K + kRankTile - 1) / kRankTile);
    if (K > 0) {
      lowrank_partial_kernel<R><<<dim3(lr_nblk, tiles), kBlock, 0, stream>>>(X, K, N, v.cs_in, ldv, lr_part, st, v.check_state && KIND >= 2);
      lowrank_reduce_kernel<R><<<1, kBlock, 0, stream>>>(lr_part, lr_nblk, K, w, lr_G, st, v.check_state && KIND >= 2);
    }
    const unsigned grid = (unsigned)((N + kBlock - 1) / kBlock);
    lowrank_expand_kernel<R, KIND><<<grid, kBlock, 0, stream>>>(X, K, lr_G, v);
  }

  int rebuild_rows() const { return K == 5 ? (sizeof(R) == 4 ? 16 : 8) : K <= 8 ? 8 : 4; }
  template <int KIND> void launch_rebuild(const Vecs<R> &v) {
    RebuildArgs<R> a;
    a.XT = XT;
    a.w = w;
    a.K = K;
    a.v = v;
    const int rows = rebuild_rows();
    const unsigned grid = (unsigned)((N + rows - 1) / rows);
    if (K == 5) rebuild_stage_kernel<R, sizeof(R) == 4 ? 16 : 8, KIND, 5, true><<<grid, kBlock, 0, stream>>>(a);
    else if (K <= 8) rebuild_stage_kernel<R, 8, KIND, 8, false><<<grid, kBlock, 0, stream>>>(a);
    else rebuild_stage_kernel<R, 4, KIND, 16, false><<<grid, kBlock, 0, stream>>>(a);
  }

  template <int KIND> void launch_kind(const Vecs<R> &v) {
    if (factored == KMT_LOWRANK_REBUILD) launch_rebuild<KIND>(v);
    else if (factored) launch_factored<KIND>(v);
    else launch_dense<KIND>(v);
  }

  void launch_by_kind(int kind, const Vecs<R> &v) {
    switch (kind) {
      case 0: launch_kind<0>(v); break;
      case 1: launch_kind<1>(v); break;
      case 2: launch_kind<2>(v); break;
      case 3: launch_kind<3>(v); break;
      case 4: launch_kind<4>(v); break;
      case 5: launch_kind<5>(v); break;
      case 6: launch_kind<6>(v); break;
      default: launch_kind<7>(v); break;
    }
  }

  int n_parts_stage7() const {
    if (factored == KMT_LOWRANK_REBUILD) return (int)((N + rebuild_rows() - 1) / rebuild_rows());
    if (factored) return lr_fused() ? lr_blocks : (int)((N + kBlock - 1) / kBlock);
    if (sym()) return (int)sym_nb;
    if (tune_bal) return bal_grid;
    return (int)((N + error_rows() - 1) / error_rows());
  }

  // Autotuner of the dense stage kernel: rows per workgroup {4, 8, 16} x
  // non-temporal adjacency loads {off, on} x grid {one workgroup per row
  // group (with and without the chunk ring), balanced: one resident round
  // with contiguous equal row ranges}, each timed on this context's own
  // matrix (stage 3 on scratch buffers).
  // Every variant sums each row in the same order (the RHS is bit-identical),
  // but the stage-7 error partials follow the variant's workgroups, so the
  // last bits of the error norm and of h can differ from the default rule's:
  // a context tuned here does not restart bit-exactly against one that was
  // not (or that picked another variant).
  int autotune(int reps) {
    if (factored || !A || sym()) return KMT_OK;  // one form of the symmetric kernels
    if (!k_scr) {
      HIP_TRY(hipMalloc((void **)&k_scr, sizeof(R) * 7 * ldv));
      HIP_TRY(hipMemsetAsync(k_scr, 0, sizeof(R) * 7 * ldv, stream));
    }
    Vecs<R> v = vecs(cs[0], cs_scr, 0);
    for (int j = 0; j < 7; ++j) v.k[j] = k_scr + j * ldv;
    hipEvent_t e0, e1;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    const int rows_opts[3] = {4, 8, 16};
    double best = 1e30;
    int best_rows = 8, best_nt = 1, best_bal = 0, best_ring = 0, best_grid = 0;
    // one workgroup per group is timed with and without the chunk ring; its
    // table entry is the faster of the two
    for (int ri = 0; ri < 3; ++ri)
      for (int nt = 0; nt < 2; ++nt)
      for (int bal = 0; bal < 2; ++bal) {
        tune_ms[ri * 4 + nt * 2 + bal] = 1e30;
        for (int ring = 0; ring < (bal ? 1 : 2); ++ring) {
          tune_rows = rows_opts[ri];
          tune_nt = nt;
          tune_bal = bal;
          tune_ring = ring;
          bal_grid = 0;
          launch_by_kind(3, v);
          HIP_TRY(hipEventRecord(e0, stream));
          for (int r = 0; r < reps; ++r) launch_by_kind(3, v);
          HIP_TRY(hipEventRecord(e1, stream));
          HIP_TRY(hipEventSynchronize(e1));
          float ms = 0;
          HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
          tune_ms[ri * 4 + nt * 2 + bal] = std::min(tune_ms[ri * 4 + nt * 2 + bal], (double)ms / reps);
          if (ms < best) {
            best = ms;
            best_rows = tune_rows;
            best_nt = nt;
            best_bal = bal;
            best_ring = ring;
            best_grid = bal_grid;
          }
        }
      }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    tune_rows = best_rows;
    tune_nt = best_nt;
    tune_bal = best_bal;
    tune_ring = best_ring;
    bal_grid = best_grid;
    tuned = 1;
    // the timed form is for right-hand sides only where attempts have a
    // faster one (N = 200 FP32: 16 us against 32 per attempt)
    pinned = !small_size();
    drop_graphs();
    return KMT_OK;
  }

  EmitArgs<R> emit_args() {
    EmitArgs<R> e;
    e.st = st;
    e.N = N;
    e.ldv = ldv;
    e.y = y;
    e.ylast = ylast;
    e.ynew = ynew;
    for (int j = 0; j < 7; ++j) e.k[j] = k[j];
    e.cs_out = cs[0];
    e.t_eval = t_eval;
    e.ring = keep_rows ? ring : nullptr;
    e.ord_part = ord_part;
    return e;
  }

  // One attempt: stages 2..7 (cs ping-pong 0->1->0->1->0->1), control,
  // emit/commit (writes stage-2 vector into cs[0]).
  void launch_attempt(std::vector<std::pair<hipEvent_t, hipEvent_t>> *ev = nullptr) {
    if (lr_path()) launch_lr_attempt(ev);
    else for (int s = 2; s <= 7; ++s) {
      const R *in = cs[(s - 2) & 1];
      R *out = cs[(s - 1) & 1];
      Vecs<R> v = vecs(in, out, 1);
      if (ev) (void)hipEventRecord((*ev)[0].first, stream);
      launch_by_kind(s, v);
      if (ev) {
        (void)hipEventRecord((*ev)[0].second, stream);
        ev->erase(ev->begin());
      }
    }
    control_kernel<R><<<1, kBlock, 0, stream>>>(st, err_part, n_parts_stage7(), N, t_eval, times, ord_part,
                                                nblk_emit, r_ring);
    launch_emit();
  }
  void launch_emit() {
    if (lr_path())
      lr_dispatch([&](auto kt, auto exact) {
        lowrank_emit_kernel<R, decltype(kt)::value, decltype(exact)::value>
            <<<lr_grid(), lr_threads(), 0, stream>>>(emit_args(), lr_args(0, 0), nblk_emit);
      });
    else if (sign_path() && K > 0)
      sign_emit_kernel<R><<<(unsigned)nblk_emit, kBlock, 0, stream>>>(emit_args(), s_pass[0].bfrag);
    else
      emit_commit_kernel<R><<<(unsigned)nblk_emit, kBlock, 0, stream>>>(emit_args());
  }
  // Before the first attempt after a change of coupling: what its paths keep
  // of the pending stage-2 vector (the low-rank partials, the signs' digits)
  void launch_prepare() {
    if (lr_path()) launch_gram(cs[0], 0);
    if (sign_path()) launch_sign_limbs(cs[0], s_pass[0].bfrag);
  }
  // the order parameters of the last attempt's rows (earlier ones are
  // computed by the next attempt's control_kernel): before the host looks
  void launch_finalize() { finalize_kernel<R><<<1, kBlock, 0, stream>>>(st, ord_part, nblk_emit, N, r_ring); }

  // Small dense networks in the working precision: whole attempts in one
  // workgroup, as far as its registers hold the matrix.  A caller's own
  // choice of stage variant (kmt_select_variant) keeps the launched kernels.
  bool small_size() const { return !factored && A && storage == KMT_ADJ_NATIVE && N <= kSmallMaxN<R>; }
  bool small_path() const { return small_size() && !pinned; }
  template <int G> void launch_small(const SmallArgs<R> &a, int n) {
    if constexpr (G < kSmallMaxGroups<R>) {
      if (N > (long)G * 8 * kSmallWaves) {
        launch_small<G + 1>(a, n);
        return;
      }
    }
    small_attempts_kernel<R, G><<<1, kSmallThreads, 0, stream>>>(a, n);
  }
  // n attempts of the run
  int launch_attempts(int n) {
    KMT_TRY(still_coupled());
    ensure_variant();
    if (small_path()) {
      SmallArgs<R> a;
      a.A = (const R *)A;
      a.lda = lda;
      a.N = N;
      a.ldv = ldv;
      a.omega = omega;
      a.y = y;
      a.ylast = ylast;
      a.ynew = ynew;
      for (int j = 0; j < 7; ++j) a.k[j] = k[j];
      a.cs = cs[0];
      a.c1 = c1;
      a.st = st;
      a.t_eval = t_eval;
      a.times = times;
      a.ring = keep_rows ? ring : nullptr;
      a.r_ring = r_ring;
      launch_small<1>(a, n);
      HIP_TRY(hipGetLastError());
      return KMT_OK;
    }
    if (!graphs_valid) KMT_TRY(build_graphs());
    for (; n >= 8; n -= 8) HIP_TRY(hipGraphLaunch(g8, stream));
    for (; n > 0; --n) HIP_TRY(hipGraphLaunch(g1, stream));
    return KMT_OK;
  }

  int build_graphs() {
    drop_graphs();
    launch_prepare();
    for (int which = 0; which < 2; ++which) {
      const int n = which == 0 ? 1 : 8;
      hipGraph_t g = nullptr;
      HIP_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
      for (int a = 0; a < n; ++a) launch_attempt();
      launch_finalize();
      HIP_TRY(hipStreamEndCapture(stream, &g));
      hipGraphExec_t ex = nullptr;
      hipError_t e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      if (e != hipSuccess) return fail(KMT_ERR_HIP, "hipGraphInstantiate failed: %s", hipGetErrorString(e));
      if (which == 0) g1 = ex;
      else g8 = ex;
    }
    graphs_valid = true;
    return KMT_OK;
  }

  // ---------------- model evaluations ----------------
  int rhs(const void *th, void *f, void *cpl) override {
    if (!coupling_ready()) return fail(KMT_ERR_STATE, "no adjacency: call kmt_set_adjacency, kmt_build_adjacency or kmt_set_factor + kmt_use_factored");
    ensure_variant();
    HIP_TRY(hipMemcpyAsync(vec_scr, th, sizeof(R) * N, hipMemcpyHostToDevice, stream));
    sincos_kernel<R><<<(unsigned)((N + kBlock - 1) / kBlock), kBlock, 0, stream>>>(vec_scr, N, ldv, cs_scr);
    Vecs<R> v = vecs(cs_scr, nullptr, 0);
    v.f_out = f_scr;
    v.cs_pairs = pairs;
    launch_by_kind(f ? KIND_RHS : KIND_COUPLING, v);
    HIP_TRY(hipGetLastError());
    if (f) HIP_TRY(hipMemcpyAsync(f, f_scr, sizeof(R) * N, hipMemcpyDeviceToHost, stream));
    if (cpl) HIP_TRY(hipMemcpyAsync(cpl, pairs, sizeof(R) * 2 * N, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  // kmt_rhs on device vectors: theta, f and the couplings stay where the
  // caller keeps them, the (cos, sin) vector goes to the caller's buffer cs
  // (rhs_scratch_bytes(), zero past N), and the launches go to stream s
  // (nullptr: the context's stream) without a synchronisation.  Nothing is
  // allocated; the factored path uses the context's partial-sum buffers.
  int rhs_device(const void *th, void *f, void *cpl, void *cs, hipStream_t s) override {
    if (!coupling_ready()) return fail(KMT_ERR_STATE, "no adjacency: call kmt_set_adjacency, kmt_build_adjacency or kmt_set_factor + kmt_use_factored");
    ensure_variant();
    const hipStream_t own = stream;
    stream = s ? s : own;
    sincos_pad_kernel<R><<<(unsigned)((ldv + kBlock - 1) / kBlock), kBlock, 0, stream>>>((const R *)th, N, ldv, (R *)cs);
    Vecs<R> v = vecs((const R *)cs, nullptr, 0);
    v.f_out = (R *)f;
    v.cs_pairs = (R *)cpl;
    launch_by_kind(f ? KIND_RHS : KIND_COUPLING, v);
    stream = own;
    HIP_TRY(hipGetLastError());
    return KMT_OK;
  }
  size_t rhs_scratch_bytes() const override { return sizeof(R) * 2 * (size_t)ldv; }
  int device_index() const override { return device; }

  int order(const void *th, double *r) override {
    HIP_TRY(hipMemcpyAsync(vec_scr, th, sizeof(R) * N, hipMemcpyHostToDevice, stream));
    const int nb = (int)((N + kBlock - 1) / kBlock);
    order_partial_kernel<R><<<nb, kBlock, 0, stream>>>(vec_scr, N, ord_scr);
    order_final_kernel<R><<<1, kBlock, 0, stream>>>(ord_scr, nb, N, ord_scr + 2 * nb);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(r, ord_scr + 2 * nb, sizeof(double), hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  // ---------------- integration ----------------
  int begin(const double *te, int ne, double t1, int keep, int rcap) override {
    if (!coupling_ready()) return fail(KMT_ERR_STATE, "no adjacency: call kmt_set_adjacency, kmt_build_adjacency or kmt_set_factor + kmt_use_factored");
    if (ne < 0) return fail(KMT_ERR_ARG, "n_eval < 0");
    if (rcap < 1) return fail(KMT_ERR_ARG, "ring_rows must be >= 1");
    HIP_TRY(hipStreamSynchronize(stream));
    drop_graphs();
    begun = 0;  // no run if the rest fails: its buffers are replaced one by one
    if (t_eval) { (void)hipFree(t_eval); t_eval = nullptr; }
    if (ring) { (void)hipFree(ring); ring = nullptr; }
    if (r_ring) { (void)hipFree(r_ring); r_ring = nullptr; }
    if (times) { (void)hipFree(times); times = nullptr; }
    if (ord_part) { (void)hipFree(ord_part); ord_part = nullptr; }
    n_eval = ne;
    keep_rows = keep;
    ring_cap = rcap;
    nblk_emit = (int)((N + kBlock - 1) / kBlock);
    std::vector<R> ter(std::max(ne, 1));
    for (int q = 0; q < ne; ++q) ter[q] = (R)te[q];
    HIP_TRY(hipMalloc((void **)&t_eval, sizeof(R) * ter.size()));
    HIP_TRY(hipMemcpyAsync(t_eval, ter.data(), sizeof(R) * ter.size(), hipMemcpyHostToDevice, stream));
    if (keep) {
      hipError_t e = hipMalloc((void **)&ring, sizeof(R) * (size_t)ring_cap * ldv);
      if (e != hipSuccess) return fail(KMT_ERR_MEMORY, "cannot allocate the output ring (%d rows): %s", ring_cap, hipGetErrorString(e));
    }
    HIP_TRY(hipMalloc((void **)&r_ring, sizeof(R) * ring_cap));
    HIP_TRY(hipMalloc((void **)&times, sizeof(R) * 2 * times_cap));
    HIP_TRY(hipMalloc((void **)&ord_part, sizeof(double) * 2 * (size_t)ring_cap * nblk_emit));
    // state
    std::memset(&shadow, 0, sizeof(shadow));
    shadow.t = t0_;
    shadow.h = h0_;
    shadow.t_last = t0_;
    shadow.t1 = (R)t1;
    shadow.atl = atl;
    shadow.rtl = rtl;
    shadow.fixed = fixed;
    shadow.active = (t0_ < (R)t1) ? 1 : 0;
    shadow.n_eval = ne;
    shadow.ring_cap = ring_cap;
    shadow.times_cap = times_cap;
    shadow.rhs_evals = 1;
    shadow.job_mode = shadow.active ? JOB_STAGE2 : JOB_NONE;
    KMT_TRY(push_state());
    ensure_variant();
    // k1 = f(y) (dp45.cu:151), then the first stage-2 vector
    sincos_kernel<R><<<(unsigned)((N + kBlock - 1) / kBlock), kBlock, 0, stream>>>(y, N, ldv, cs[1]);
    Vecs<R> v = vecs(cs[1], nullptr, 0);
    v.f_out = k[0];
    launch_by_kind(KIND_RHS, v);
    launch_emit();
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(stream));
    begun = 1;
    return KMT_OK;
  }

  void fill_status(kmt_status *s) {
    if (!s) return;
    s->t = (double)shadow.t;
    s->h = (double)shadow.h;
    s->t_last = (double)shadow.t_last;
    s->accepted = (long)shadow.accepted;
    s->rejected = (long)shadow.rejected;
    s->attempts = (long)shadow.attempts;
    s->rhs_evals = (long)shadow.rhs_evals;
    s->active = shadow.active;
    s->error = shadow.error;
    s->rows_ready = shadow.ring_count;
    s->times_ready = shadow.times_count;
    s->eval_i = shadow.eval_i;
    s->pending = shadow.commit_pending ? shadow.pend_hi - shadow.pend_lo : 0;
  }

  int advance(int max_attempts, kmt_status *s) override {
    if (!begun) return fail(KMT_ERR_STATE, "kmt_advance before kmt_begin");
    if (max_attempts < 0) return fail(KMT_ERR_ARG, "max_attempts < 0");
    KMT_TRY(fetch_state());
    int n = std::min(max_attempts, shadow.times_cap - shadow.times_count);
    if (shadow.active && n > 0) {
      KMT_TRY(flush_state());
      KMT_TRY(launch_attempts(n));
    }
    KMT_TRY(fetch_state());
    fill_status(s);
    if (shadow.error) return fail(KMT_ERR_NUMERIC, "error norm is not finite at t=%g (h=%g): integration stopped", (double)shadow.t, (double)shadow.h);
    return KMT_OK;
  }

  // cpl (optional): the couplings (C_i, S_i) of every drained row, 2N values
  // a row, computed from the row where it sits in the ring (the launches of
  // kmt_rhs's coupling form, one row at a time through the shared (cos, sin)
  // and pair buffers, each copied out before the next row overwrites them).
  int read_outputs(int max_rows, void *rows, void *rv, void *cpl, int *nout) override {
    if (!begun) return fail(KMT_ERR_STATE, "kmt_read_outputs before kmt_begin");
    KMT_TRY(fetch_state());
    const int ready = shadow.ring_count;
    const int n = std::min(std::max(max_rows, 0), ready);
    if ((rows || cpl) && n > 0 && !keep_rows) return fail(KMT_ERR_STATE, "rows were not kept (kmt_begin keep_rows=0)");
    if (cpl && n > 0 && !coupling_ready()) return fail(KMT_ERR_STATE, "no adjacency for the couplings");
    if (ready == 0) {
      if (nout) *nout = 0;
      return KMT_OK;
    }
    if (rows && n > 0) KMT_TRY(drain_rows(rows, ring, sizeof(R) * ldv, sizeof(R) * N, n));
    if (cpl && n > 0) ensure_variant();
    for (int q = 0; cpl && q < n; ++q) {
      sincos_kernel<R><<<(unsigned)((N + kBlock - 1) / kBlock), kBlock, 0, stream>>>(ring + (size_t)q * ldv, N, ldv, cs_scr);
      Vecs<R> v = vecs(cs_scr, nullptr, 0);
      v.f_out = f_scr;
      v.cs_pairs = pairs;
      launch_by_kind(KIND_COUPLING, v);
      HIP_TRY(hipGetLastError());
      HIP_TRY(hipMemcpyAsync((R *)cpl + (size_t)q * 2 * N, pairs, sizeof(R) * 2 * N, hipMemcpyDeviceToHost, stream));
    }
    if (rv && n > 0) HIP_TRY(hipMemcpyAsync(rv, r_ring, sizeof(R) * n, hipMemcpyDeviceToHost, stream));
    // keep the unread rows at the front of the ring (in order)
    for (int q = n; q < ready; ++q) {
      if (keep_rows) HIP_TRY(hipMemcpyAsync(ring + (size_t)(q - n) * ldv, ring + (size_t)q * ldv, sizeof(R) * N, hipMemcpyDeviceToDevice, stream));
      HIP_TRY(hipMemcpyAsync(r_ring + (q - n), r_ring + q, sizeof(R), hipMemcpyDeviceToDevice, stream));
    }
    shadow.ring_count = ready - n;
    dirty = true;
    HIP_TRY(hipStreamSynchronize(stream));
    if (nout) *nout = n;
    return KMT_OK;
  }

  int read_times(int max_n, void *tv, void *hv, int *nout) override {
    if (!begun) return fail(KMT_ERR_STATE, "kmt_read_times before kmt_begin");
    KMT_TRY(fetch_state());
    const int ready = shadow.times_count;
    const int n = std::min(std::max(max_n, 0), ready);
    if (ready > 0) {
      std::vector<R> buf(2 * ready);
      HIP_TRY(hipMemcpyAsync(buf.data(), times, sizeof(R) * 2 * ready, hipMemcpyDeviceToHost, stream));
      HIP_TRY(hipStreamSynchronize(stream));
      for (int q = 0; q < n; ++q) {
        if (tv) ((R *)tv)[q] = buf[2 * q];
        if (hv) ((R *)hv)[q] = buf[2 * q + 1];
      }
      if (n > 0 && n < ready) {
        HIP_TRY(hipMemcpyAsync(times, buf.data() + 2 * n, sizeof(R) * 2 * (ready - n), hipMemcpyHostToDevice, stream));
        HIP_TRY(hipStreamSynchronize(stream));
      }
      shadow.times_count = ready - n;
      dirty = true;
    }
    if (nout) *nout = n;
    return KMT_OK;
  }

  int step(int *acc, double *t, double *h) override {
    if (!begun) return fail(KMT_ERR_STATE, "kmt_step before kmt_begin");
    KMT_TRY(fetch_state());
    const long long before = shadow.accepted;
    if (shadow.active && shadow.times_count < shadow.times_cap) {
      KMT_TRY(flush_state());
      KMT_TRY(launch_attempts(1));
    }
    KMT_TRY(fetch_state());
    if (acc) *acc = shadow.accepted > before ? 1 : 0;
    if (t) *t = (double)shadow.t;
    if (h) *h = (double)shadow.h;
    if (shadow.error) return fail(KMT_ERR_NUMERIC, "error norm is not finite at t=%g", (double)shadow.t);
    return KMT_OK;
  }

  int eval(double te, void *out) override {
    if (!begun) return fail(KMT_ERR_STATE, "kmt_eval before kmt_begin");
    interp_kernel<R><<<(unsigned)((N + kBlock - 1) / kBlock), kBlock, 0, stream>>>(st, N, ylast, k[0], k[1], k[2], k[3], k[4], k[5], k[6], (R)te, vec_scr);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(out, vec_scr, sizeof(R) * N, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  // ---------------- timing ----------------
  int time_stage(int reps, double *avg_ms) override {
    if (!coupling_ready()) return fail(KMT_ERR_STATE, "no adjacency");
    if (reps < 1) return fail(KMT_ERR_ARG, "reps < 1");
    ensure_variant();
    hipEvent_t e0, e1;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    // stage 3 on scratch k buffers (the integrator's k_j stay untouched)
    if (!k_scr) {
      HIP_TRY(hipMalloc((void **)&k_scr, sizeof(R) * 7 * ldv));
      HIP_TRY(hipMemsetAsync(k_scr, 0, sizeof(R) * 7 * ldv, stream));
    }
    Vecs<R> v = vecs(cs[0], cs_scr, 0);
    for (int j = 0; j < 7; ++j) v.k[j] = k_scr + j * ldv;
    launch_by_kind(3, v);  // warm
    HIP_TRY(hipEventRecord(e0, stream));
    for (int r = 0; r < reps; ++r) launch_by_kind(3, v);
    HIP_TRY(hipEventRecord(e1, stream));
    HIP_TRY(hipEventSynchronize(e1));
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (avg_ms) *avg_ms = ms / reps;
    return KMT_OK;
  }

  int time_attempts(int attempts, double *region_ms, double *stage_avg_ms, kmt_status *s) override {
    if (!begun) return fail(KMT_ERR_STATE, "kmt_time_attempts before kmt_begin");
    if (attempts < 1) return fail(KMT_ERR_ARG, "attempts < 1");
    KMT_TRY(fetch_state());
    if (attempts > shadow.times_cap - shadow.times_count)
      return fail(KMT_ERR_ARG, "attempts exceed the accepted-step log capacity; drain kmt_read_times first");
    KMT_TRY(still_coupled());
    ensure_variant();
    const bool launches = !small_path();  // the one-workgroup form has no stage launches to time
    std::vector<std::pair<hipEvent_t, hipEvent_t>> pairs_all(launches ? 6 * attempts : 0);
    for (auto &p : pairs_all) {
      HIP_TRY(hipEventCreate(&p.first));
      HIP_TRY(hipEventCreate(&p.second));
    }
    hipEvent_t r0, r1;
    HIP_TRY(hipEventCreate(&r0));
    HIP_TRY(hipEventCreate(&r1));
    std::vector<std::pair<hipEvent_t, hipEvent_t>> work = pairs_all;
    KMT_TRY(flush_state());
    if (launches) launch_prepare();
    HIP_TRY(hipEventRecord(r0, stream));
    if (launches) {
      for (int a = 0; a < attempts; ++a) launch_attempt(&work);
      launch_finalize();
    } else {
      KMT_TRY(launch_attempts(attempts));
    }
    HIP_TRY(hipEventRecord(r1, stream));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipEventSynchronize(r1));
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, r0, r1));
    double tot = 0;
    for (auto &p : pairs_all) {
      float m = 0;
      HIP_TRY(hipEventElapsedTime(&m, p.first, p.second));
      tot += m;
      (void)hipEventDestroy(p.first);
      (void)hipEventDestroy(p.second);
    }
    (void)hipEventDestroy(r0);
    (void)hipEventDestroy(r1);
    if (region_ms) *region_ms = ms;
    if (stage_avg_ms) *stage_avg_ms = launches ? tot / pairs_all.size() : ms / (6 * attempts);
    KMT_TRY(fetch_state());
    fill_status(s);
    if (shadow.error) return fail(KMT_ERR_NUMERIC, "error norm is not finite");
    return KMT_OK;
  }
};


EngineBase *new_engine_f32();
EngineBase *new_engine_f64();

}  // namespace kmt
