// Host driver of a full Lloyd fit (src/kmeans_lloyd_driver.hpp:21-431).
//
// Semantics kept from the reference: iterate while it < max_iter and the sum
// of squared centroid shifts, compared in the data type, exceeds tol (raw, not
// variance-scaled); each iteration computes half-norms, the fused
// assignment+update, the reduction of private copies with the empty-cluster
// list, the relocation of empty clusters (on unnormalised sums, before the
// division), the division, the shifts and their sum; the epilogue recomputes
// labels and the weighted inertia of the final centroids and copies them to
// res_centroids_t.  init_centroids_t is one of the rotating centroid buffers
// and is overwritten.
//
// Differences (all on the host side, none in results):
//  * the host is off the GPU's critical path: an iteration is three launches
//    (step, reduction, tail), enqueued without a host decision.  The tail
//    kernel keeps the loop's state on the device (finished iterations, and
//    whether the loop converged or found empty clusters) and publishes it in
//    pinned host memory; the kernels of an iteration return at once when the
//    loop has stopped, so the next iteration is enqueued ahead and costs next
//    to nothing when it was not needed.  The host reads the state from
//    memory between launches; it relocates empty clusters and enqueues the
//    iterations after that again;
//  * private copies are one per block of the persistent fused kernel and are
//    written with plain stores, so the sums are deterministic (not on the two
//    paths that add the blocks' totals into eight copies with atomics: float32
//    beyond the tiled kernels, d > 128 or k > 32768, and sums that do not fit
//    LDS on the generic one; there the last bits depend on the blocks' order);
//  * the relocation path reuses the labels of the fused step instead of
//    recomputing them from the same centroids and half-norms
//    (src/kmeans_lloyd_driver.hpp:226-250);
//  * the verbose line reports the inertia of the centroids that produced the
//    labels (the reference evaluates it against the undivided sums).
#include <cstdlib>
#include <cstring>
#include <exception>
#include <map>
#include <memory>
#include <mutex>
#include <sstream>
#include <thread>
#include <tuple>
#include <vector>

#include "common.hpp"
#include "lloyd_fast.hpp"

namespace kmd {

// A part of one allocation.
struct Slice {
  char *ptr = nullptr;
  size_t size = 0;
  template <typename U>
  U *as() const {
    return reinterpret_cast<U *>(ptr);
  }
  size_t bytes() const { return size; }
};

template <typename T, typename I>
struct LloydWorkspace {
  int64_t n, d, k;
  int blocks = 1;          // private copies / partial slots
  bool fast = false;       // MFMA fast path (fixed-point partials)
  bool store_flush = false;
  int mixed_terms = 0;     // BF16 split terms (1 or 3) or 8 (FP8) of the mixed path, 0: FP32
  bool tiled = false;      // tiled path: centroids streamed, separate update
  bool wide = false;       // features streamed, separate update (d > 128)
  int blocks_b = 0;        // partial slots of the FP32 re-score (mixed path)
  // LDS-resident mixed path: the re-score restricted to candidate tiles,
  // from the sample-major copy xr, and the queue's separate exact update
  bool mixed_cand = false;
  // LDS-resident mixed path: undecided samples re-scored inside the kernel
  bool mixed_ink = false;
  FusedPlan plan;
  // one allocation for what every path has (a stream-ordered allocation and
  // its release cost several microseconds of host time each)
  TempBuffer arena{0, nullptr};
  Slice hn, sizes, shifts, per_sample, copies, sizes_copies, list, scalars, scales;
  Slice stats;   // of the fixed-point scales
  TempBuffer aop{0, nullptr}, bound{0, nullptr}, queue{0, nullptr},
      queue_counts{0, nullptr};
  TempBuffer xr{0, nullptr}, upd{0, nullptr};  // tiled: X sample-major, update scratch
  TempBuffer qmask{0, nullptr}, cand{0, nullptr};  // tiled BF16: candidate tiles
  TempBuffer xb{0, nullptr}, xnb{0, nullptr};  // tiled BF16 (T = 1): BF16 samples
  int64_t seg_cap = 0;     // capacity of each block's re-score queue segment
  // `sums`: the undivided sums of the iteration (kept until the next one's
  // reduction, for the relocation of empty clusters); `scalars`: the loop's
  // state @0, an iteration's re-scored count @48, the epilogue's sum @56
  Slice sums, tail_part, tail_ticket;
  // copies_bytes / sizes_bytes: private copies of the generic kernel, or the
  // fast path's per-block partials (in `copies`, sizes_bytes = 0)
  LloydWorkspace(int64_t n_, int64_t d_, int64_t k_, int blocks_, bool fast_,
                 bool store_, const FusedPlan &plan_, size_t copies_bytes,
                 size_t sizes_bytes, hipStream_t s)
      : n(n_), d(d_), k(k_), blocks(blocks_), fast(fast_), store_flush(store_),
        plan(plan_) {
    size_t used = 0;
    auto take = [&](Slice &q, size_t bytes) {
      q.ptr = reinterpret_cast<char *>(used);   // offset, until the base is known
      q.size = bytes;
      used += (bytes + 255) / 256 * 256;
    };
    Slice *const all[] = {&scalars, &tail_ticket, &hn,   &sizes,     &shifts, &list,
                          &scales,  &stats,       &sums, &tail_part, &per_sample,
                          &copies,  &sizes_copies};
    take(scalars, 64);
    take(tail_ticket, 64);
    take(hn, sizeof(T) * k_);
    take(sizes, sizeof(T) * k_);
    take(shifts, sizeof(T) * k_);
    take(list, sizeof(I) * (k_ + 1));
    take(scales, fast_ ? sizeof(float) * (d_ + 1) + 16 : 0);
    take(stats, fast_ ? fixed_point_stats_bytes(d_) : 0);
    take(sums, sizeof(T) * d_ * k_);
    take(tail_part, sizeof(double) * step_tail_partials(k_));
    take(per_sample, sizeof(T) * (n_ > 0 ? n_ : 1));
    take(copies, copies_bytes);
    take(sizes_copies, sizes_bytes);
    arena = TempBuffer(used, s);
    for (Slice *q : all) q->ptr = arena.as<char>() + reinterpret_cast<size_t>(q->ptr);
    // scalars and the ticket lie at the front
    KMD_HIP_CHECK(hipMemsetAsync(arena.as<char>(), 0, 512, s));
  }
  LoopState *state() const { return scalars.as<LoopState>(); }
  const int *stop() const { return &state()->stop; }
  int *queue_count() const {
    static_assert(sizeof(LoopState) <= 48, "layout of scalars");
    return reinterpret_cast<int *>(scalars.as<char>() + 48);
  }
  double *epilogue_sum() const {
    return reinterpret_cast<double *>(scalars.as<char>() + 56);
  }
  float *scale() const { return scales.as<float>(); }
  int *nonfinite() const {
    return reinterpret_cast<int *>(scales.as<char>() + sizeof(float) * (d + 1));
  }
};

// Re-score forms of the LDS-resident mixed path.  By default undecided
// samples are re-scored inside the BF16 kernel (when the FP32 centroid tiles
// fit LDS beside its own data), else by a second kernel that gathers every
// queued sample over all tiles and adds it to the sums.
// KMD_MIXED_GATHER=1 keeps the second kernel; KMD_MIXED_CAND=1 switches to
// the candidate-tile re-score from a sample-major copy of X plus a separate
// exact update of the queue (fewer bytes per queued sample, four more
// launches per iteration; at n = 10M, d = 32, k = 256: 630 iters/s against
// the gather's 795).
static bool env_is_1(const char *name) {
  const char *e = std::getenv(name);
  return e != nullptr && e[0] == '1';
}
static bool mixed_cand_requested() { return env_is_1("KMD_MIXED_CAND"); }
static bool mixed_gather_requested() { return env_is_1("KMD_MIXED_GATHER"); }

// Mixed-precision workspace: BF16 kernel partials, then FP32 re-score
// partials; returns nullptr when the shape is not served or the inputs hold
// non-finite values (the FP32 path handles those).
template <typename T, typename I>
static std::unique_ptr<LloydWorkspace<T, I>> make_mixed_workspace(
    int64_t n, int64_t d, int64_t k, int terms, const T *X, const T *w,
    hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    if (n <= 0 || !fast_fused_supported<T>(d, k)) return nullptr;
    // candidate tiles: the re-score of an undecided sample covers only the
    // 32-centroid tiles whose BF16 best is within the bound of its best,
    // reading the sample from a sample-major copy of X (made once per fit)
    const bool cand = tiled_cand_supported(k) && tiled_supported(d, k) &&
                      mixed_cand_fits(d, k, terms) && mixed_cand_requested();
    const bool ink = !cand && !mixed_gather_requested() && mixed_ink_fits(d, k, terms);
    const int ba = mixed_blocks<I>(n, d, k, terms, cand, ink);
    const int bb = ink ? 0 : fast_rescore_blocks<I>(d, k, ba);
    if (ba < 1 || (!ink && bb < 1)) return nullptr;
    auto ws = std::make_unique<LloydWorkspace<T, I>>(
        n, d, k, ba, true, true, FusedPlan{},
        sizeof(int64_t) * (size_t)(ba + bb) * (d * k + k), 0, s);
    ws->mixed_terms = terms;
    ws->mixed_ink = ink;
    ws->blocks_b = bb;
    ws->aop = TempBuffer(mixed_aop_bytes(d, k, terms), s);
    ws->bound = TempBuffer(2 * sizeof(float), s);
    ws->seg_cap = ink ? 0 : mixed_seg_cap(n, d, ba);
    ws->queue = TempBuffer(sizeof(int) * (size_t)ba * ws->seg_cap, s);
    ws->queue_counts = TempBuffer(sizeof(int) * (size_t)ba, s);
    launch_fixed_point_scales(n, d, X, w, ws->scale(), ws->nonfinite(), s,
                              ws->stats.template as<void>());
    int bad = 0;
    KMD_HIP_CHECK(hipMemcpyAsync(&bad, ws->nonfinite(), sizeof(int),
                                 hipMemcpyDeviceToHost, s));
    KMD_HIP_CHECK(hipStreamSynchronize(s));
    if (bad) return nullptr;
    if (cand) {
      ws->mixed_cand = true;
      ws->qmask = TempBuffer(sizeof(unsigned) * (size_t)ba * ws->seg_cap, s);
      ws->cand = TempBuffer(tiled_cand_scratch_bytes(n, k), s);
      ws->xr = TempBuffer(sizeof(float) * (size_t)n * d, s);
      launch_transpose(n, d, X, ws->xr.template as<float>(), s);
    }
    return ws;
  } else {
    (void)n, (void)d, (void)k, (void)terms, (void)X, (void)w, (void)s;
    return nullptr;
  }
}

// Tiled workspace (float, finite inputs): X_r, one int64 sum slot, update
// scratch; with precision != FP32 also the BF16 operands and queue.  Returns
// nullptr for non-finite inputs (the generic path propagates them).
template <typename T, typename I>
static std::unique_ptr<LloydWorkspace<T, I>> make_tiled_workspace(
    int64_t n, int64_t d, int64_t k, int precision, const T *X, const T *w,
    hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    if (n <= 0 || !tiled_supported(d, k)) return nullptr;
    auto ws = std::make_unique<LloydWorkspace<T, I>>(
        n, d, k, 1, true, true, FusedPlan{}, sizeof(int64_t) * (size_t)(d * k + k),
        0, s);
    launch_fixed_point_scales(n, d, X, w, ws->scale(), ws->nonfinite(), s,
                              ws->stats.template as<void>());
    int bad = 0;
    KMD_HIP_CHECK(hipMemcpyAsync(&bad, ws->nonfinite(), sizeof(int),
                                 hipMemcpyDeviceToHost, s));
    KMD_HIP_CHECK(hipStreamSynchronize(s));
    if (bad) return nullptr;
    ws->tiled = true;
    ws->xr = TempBuffer(sizeof(float) * (size_t)n * d, s);
    bool have_xr = false;
    ws->upd = TempBuffer(tiled_update_scratch_bytes(n, k), s);
    if (precision != KMD_PREC_FP32) {
      // BF16 terms, or 8: the FP8 (e4m3) kernel
      const int terms = precision == KMD_PREC_BF16X3 ? 3
                        : precision == KMD_PREC_FP8  ? 8
                                                     : 1;
      const int ba = tiled_mixed_blocks<I>(n, d, k, terms);
      if (ba >= 1) {
        ws->mixed_terms = terms;
        ws->blocks_b = ba;
        ws->seg_cap = tiled_mixed_seg_cap(n, d, terms, ba);
        ws->aop = TempBuffer(tiled_aop_bytes(d, k, terms), s);
        ws->bound = TempBuffer(sizeof(float) * tiled_bound_floats(), s);
        ws->queue = TempBuffer(sizeof(int) * (size_t)ba * ws->seg_cap, s);
        ws->queue_counts = TempBuffer(sizeof(int) * (size_t)ba, s);
        if (tiled_cand_supported(k)) {
          ws->qmask = TempBuffer(sizeof(unsigned) * (size_t)ba * ws->seg_cap, s);
          ws->cand = TempBuffer(tiled_cand_scratch_bytes(n, k), s);
        }
        if (terms == 1 || terms == 8) {
          ws->xb = TempBuffer(tiled_xb_bytes(n, d), s);
          ws->xnb = TempBuffer(sizeof(float) * (size_t)n, s);
          if (terms == 1)
            launch_tiled_xb_prep(n, d, X, ws->xr.template as<float>(),
                                 ws->xb.template as<void>(),
                                 ws->xnb.template as<float>(), s);
          else
            launch_tiled_x8_prep(n, d, X, ws->xb.template as<void>(),
                                 ws->xnb.template as<float>(),
                                 ws->bound.template as<float>(), s);
          have_xr = terms == 1;
        }
      }
    }
    if (!have_xr) launch_transpose(n, d, X, ws->xr.template as<float>(), s);
    return ws;
  } else {
    (void)n, (void)d, (void)k, (void)precision, (void)X, (void)w, (void)s;
    return nullptr;
  }
}

// ---- launch tuning ----------------------------------------------------------
// The choice in force on this thread (read by the planners while a driver
// call runs), the autotuner's table per (d, k, precision, log2 n) and a
// process-wide override (kmd_set_tuning).
namespace {
thread_local int t_blocks_cap = 0;
thread_local int t_path = 0;
thread_local int t_shape = 0;
thread_local bool t_separate = false;   // no one-block loop (while timing plans)
struct TuneChoice {
  int path = 0, blocks_per_cu = 0, shape = 0;
};
struct TuneGuard {
  int pb, pp, ps;
  explicit TuneGuard(const TuneChoice &c)
      : pb(t_blocks_cap), pp(t_path), ps(t_shape) {
    t_blocks_cap = c.blocks_per_cu;
    t_path = c.path;
    t_shape = c.shape;
  }
  ~TuneGuard() {
    t_blocks_cap = pb;
    t_path = pp;
    t_shape = ps;
  }
};
std::mutex g_tune_mu;
std::map<std::tuple<int64_t, int64_t, int, int>, TuneChoice> g_tune;
bool g_override = false;
TuneChoice g_override_choice;

int log2_bucket(int64_t n) {
  int b = 0;
  while ((int64_t(1) << (b + 1)) <= n) ++b;
  return b;
}

// A plan is for a fit of several launches: where one block does the whole fit
// (f32, small_loop_serves, which not every n of a bucket is) the table is not
// asked.
TuneChoice choose_tuning(int64_t n, int64_t d, int64_t k, int precision, bool f32) {
  TuneChoice c;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    if (g_override) return g_override_choice;
    auto it = g_tune.find(std::make_tuple(d, k, precision, log2_bucket(n)));
    if (it == g_tune.end()) return c;
    c = it->second;
  }
  return f32 && small_loop_serves(n, d, k) ? TuneChoice{} : c;
}
}  // namespace

int tuned_blocks_per_cu() { return t_blocks_cap; }
int tuned_path() { return t_path; }
int tuned_shape() { return t_shape; }

void set_tuning_override(int path, int blocks_per_cu, int shape) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_override = path >= 0;
  g_override_choice.path = path < 0 ? 0 : path;
  g_override_choice.blocks_per_cu = blocks_per_cu < 0 ? 0 : blocks_per_cu;
  g_override_choice.shape = shape < 0 ? 0 : shape;
}

// Test hook: KMD_FORCE_TILED=1 selects the tiled path for every shape it
// serves (the LDS-resident kernels are otherwise preferred).
static bool force_tiled() {
  const char *e = std::getenv("KMD_FORCE_TILED");
  return e != nullptr && e[0] == '1';
}

template <typename T, typename I>
static std::unique_ptr<LloydWorkspace<T, I>> make_workspace(int64_t n,
                                                            int64_t d,
                                                            int64_t k,
                                                            const T *X,
                                                            const T *w,
                                                            int precision,
                                                            hipStream_t s) {
  // With k <= 32 the step is bound by reading X, not by the cross term:
  // every precision runs the FP32 few-centroid kernel there (its labels and
  // sums are what the mixed paths reproduce, at a fraction of their time).
  const bool smallk = std::is_same<T, float>::value && !force_tiled() &&
                      tuned_path() != 2 && fast_smallk_serves(d, k);
  // the FP8 cross term is built on the tiled kernels only
  const bool tiled_first = !smallk && (force_tiled() || tuned_path() == 2 ||
                                       (precision == KMD_PREC_FP8 &&
                                        std::is_same<T, float>::value &&
                                        tiled_supported(d, k)));
  if (precision != KMD_PREC_FP32 && precision != KMD_PREC_FP8 && !tiled_first &&
      !smallk) {
    auto ws = make_mixed_workspace<T, I>(
        n, d, k, precision == KMD_PREC_BF16X3 ? 3 : 1, X, w, s);
    if (ws) return ws;
  }
  if (tiled_first || !fast_fused_supported<T>(d, k)) {
    auto ws = make_tiled_workspace<T, I>(n, d, k, precision, X, w, s);
    if (ws) return ws;
  }
  if (n > 0 && fast_fused_supported<T>(d, k)) {
    const int blocks = fast_fused_blocks<I>(n, d, k);
    auto ws = std::make_unique<LloydWorkspace<T, I>>(
        n, d, k, blocks, true, true, FusedPlan{},
        sizeof(int64_t) * (size_t)blocks * (d * k + k), 0, s);
    return ws;   // its fixed-point scales: driver_impl
  }
  FusedPlan p = plan_generic_fused<T>(n, d, k);
  // features streamed through the matrix core: the same sums into the same
  // copies as the generic kernel's atomics
  const bool wide = std::is_same<T, float>::value && wide_supported(n, d, k) &&
                    label_sums_supported(k);
  if (p.priv && !wide)
    return std::make_unique<LloydWorkspace<T, I>>(
        n, d, k, p.blocks, false, true, p, sizeof(T) * (size_t)p.blocks * d * k,
        sizeof(T) * (size_t)p.blocks * k, s);
  // sums too large for LDS: atomics into a few zeroed copies
  const int copies = 8;
  auto ws = std::make_unique<LloydWorkspace<T, I>>(
      n, d, k, copies, false, false, p, sizeof(T) * (size_t)copies * d * k,
      sizeof(T) * (size_t)copies * k, s);
  ws->wide = wide;
  return ws;
}

// Iterations enqueued ahead of the last one known to have finished.  One covers
// the launches of the next (50,000 x 14 x 127, 18 us of kernels an iteration: 883
// us a fit, 902 with three ahead; no fit tried was faster with three), and every
// further one is a kernel of the whole chip that other streams wait behind.
// Beside the server's engine three made a stream of 200 requests/s wait 43 ms
// (median) where one makes it 25 and none 13, and a saturated one 0.56 / 0.41 /
// 0.20 s, at 278 / 292 / 299 fits/s; a fit alone takes 1.7 % longer with none
// (2M x 96 x 512).  So a thread whose fits share the GPU can ask for none.
constexpr int kAhead = 1;
thread_local int t_run_ahead = kAhead;

int set_run_ahead(int iterations) {
  const int before = t_run_ahead;
  t_run_ahead = iterations < 0 || iterations > kAhead ? kAhead : iterations;
  return before;
}

// Optional timing of the fused-step kernel with HIP events on the driver's
// stream: one event pair per iteration that can be in flight, read back once
// that iteration is known to have finished.
struct FusedTimer {
  bool on = false;
  hipEvent_t start[kAhead + 1] = {}, stop[kAhead + 1] = {};
  int slot = 0;
  double total_ms = 0.0;
  int64_t launches = 0;
  explicit FusedTimer(bool enable) : on(enable) {
    if (on) {
      for (int i = 0; i <= kAhead; ++i) {
        KMD_HIP_CHECK(hipEventCreate(&start[i]));
        KMD_HIP_CHECK(hipEventCreate(&stop[i]));
      }
    }
  }
  ~FusedTimer() {
    for (int i = 0; i <= kAhead; ++i) {
      if (start[i]) (void)hipEventDestroy(start[i]);
      if (stop[i]) (void)hipEventDestroy(stop[i]);
    }
  }
  void begin(hipStream_t s) {
    if (on) KMD_HIP_CHECK(hipEventRecord(start[slot], s));
  }
  void end(hipStream_t s) {
    if (on) KMD_HIP_CHECK(hipEventRecord(stop[slot], s));
  }
  // the launch timed in slot i has finished
  void collect(int i) {
    if (!on) return;
    float ms = 0.f;
    KMD_HIP_CHECK(hipEventSynchronize(stop[i]));
    KMD_HIP_CHECK(hipEventElapsedTime(&ms, start[i], stop[i]));
    total_ms += ms;
    ++launches;
  }
};

// Pinned host memory for the loop's published state (LoopHost).  Pinning and
// unpinning cost hundreds of microseconds, so the 64-byte blocks are kept in
// a process-wide free list and reused (one per driver call running at a time).
std::mutex g_pinned_mu;
std::vector<char *> g_pinned_free;

struct PinnedScalars {
  char *p = nullptr;
  PinnedScalars() {
    {
      std::lock_guard<std::mutex> lk(g_pinned_mu);
      if (!g_pinned_free.empty()) {
        p = g_pinned_free.back();
        g_pinned_free.pop_back();
      }
    }
    if (p == nullptr)
      KMD_HIP_CHECK(hipHostMalloc(reinterpret_cast<void **>(&p), 64, hipHostMallocDefault));
    std::memset(p, 0, 64);
  }
  ~PinnedScalars() {
    if (p == nullptr) return;
    std::lock_guard<std::mutex> lk(g_pinned_mu);
    g_pinned_free.push_back(p);
  }
  PinnedScalars(const PinnedScalars &) = delete;
  PinnedScalars &operator=(const PinnedScalars &) = delete;
  LoopHost *host() const { return reinterpret_cast<LoopHost *>(p); }
};
static_assert(sizeof(LoopHost) <= 64, "one pinned block holds the state");

// Leaves no kernel behind that may still write the pinned block when the
// driver is left by an exception.
struct DrainOnThrow {
  hipStream_t s;
  int entered = std::uncaught_exceptions();
  ~DrainOnThrow() {
    if (std::uncaught_exceptions() > entered) (void)hipStreamSynchronize(s);
  }
};

// Waits until `host` shows more than `done` finished iterations or a stopped
// loop; its word.  A device error ends the wait.
inline unsigned long long wait_loop(const LoopHost *host, long long done, hipStream_t s) {
  auto word = [&] { return __atomic_load_n(&host->word, __ATOMIC_ACQUIRE); };
  auto ended = [&](unsigned long long w) {
    return (long long)(w >> 2) > done || (w & 3) != 0;
  };
  for (int spins = 1;; ++spins) {
    unsigned long long w = word();
    if (ended(w)) return w;
    if (spins % 4096 == 0) {
      const hipError_t e = hipStreamQuery(s);
      if (e == hipSuccess) {   // all done: the word must be there
        w = word();
        if (ended(w)) return w;
        throw RuntimeError("Lloyd loop: an iteration left no state");
      }
      if (e != hipErrorNotReady) KMD_HIP_CHECK(e);
      (void)hipGetLastError();   // "not ready" is no error of a later launch
      std::this_thread::yield();
    } else {
      __builtin_ia32_pause();
    }
  }
}

// LDS-resident mixed path: BF16 step (operands already prepared for `cur`)
// and the re-score of its undecided samples, in the workspace's form:
// labels (the FP32 path's) and the int64 partial slots.
template <typename T, typename I>
static void mixed_labels_and_partials(LloydWorkspace<T, I> &ws, const T *X,
                                      const T *w, const T *cur, I *labels,
                                      hipStream_t s, const int *skip) {
  if constexpr (std::is_same<T, float>::value) {
    const int64_t n = ws.n, d = ws.d, k = ws.k;
    launch_mixed_step<I>(n, d, k, ws.mixed_terms, ws.blocks, X, w,
                         ws.aop.template as<const void>(),
                         ws.bound.template as<const float>(), ws.scale(),
                         labels, ws.copies.template as<void>(),
                         ws.queue.template as<int>(),
                         ws.queue_counts.template as<int>(),
                         ws.mixed_cand ? ws.qmask.template as<unsigned>() : nullptr, s,
                         skip, ws.mixed_ink ? cur : nullptr,
                         ws.mixed_ink ? ws.hn.template as<const T>() : nullptr,
                         ws.mixed_ink ? ws.queue_count() : nullptr);
    if (ws.mixed_ink) {
      // re-scored inside the kernel: nothing more to launch
    } else if (ws.mixed_cand) {
      // FP32 re-score of the candidate tiles (labels), then the exact sums
      // of the re-scored samples into the re-score partial slots
      launch_tiled_cand_rescore<I>(
          n, d, k, ws.xr.template as<const float>(), cur, ws.hn.template as<const T>(),
          labels, ws.queue.template as<const int>(),
          ws.queue_counts.template as<const int>(),
          ws.qmask.template as<const unsigned>(), ws.blocks, ws.seg_cap,
          ws.cand.template as<void>(), ws.queue_count(), s, skip);
      launch_queue_update<I>(d, k, ws.blocks_b, ws.blocks, ws.seg_cap,
                             ws.queue.template as<const int>(),
                             ws.queue_counts.template as<const int>(),
                             ws.xr.template as<const float>(), w, labels, ws.scale(),
                             ws.copies.template as<int64_t>() + (size_t)ws.blocks * (d * k + k),
                             s, skip);
    } else {
      launch_fast_rescore<I>(n, d, k, X, w, cur, ws.hn.template as<const T>(),
                             labels, ws.scale(), ws.nonfinite(),
                             ws.copies.template as<void>(), ws.blocks,
                             ws.queue.template as<const int>(),
                             ws.queue_counts.template as<const int>(),
                             ws.blocks, ws.seg_cap, ws.queue_count(), s, skip);
    }
  } else {
    (void)ws, (void)X, (void)w, (void)cur, (void)labels, (void)s, (void)skip;
    throw RuntimeError("mixed-precision step: float32 only");
  }
}

// Fused step and reduction for centroids `cur` (half norms in ws.hn):
// undivided sums into ws.sums, cluster sizes into ws.sizes.
template <typename T, typename I>
static void lloyd_front(LloydWorkspace<T, I> &ws, const T *X, const T *w,
                        const T *cur, I *labels, hipStream_t s, FusedTimer &timer) {
  const int64_t n = ws.n, d = ws.d, k = ws.k;
  const int *skip = ws.stop();
  T *sums = ws.sums.template as<T>();
  T *sizes = ws.sizes.template as<T>();
  auto reduce_fixed = [&](int64_t slots) {
    launch_sum_fixed_partials<T>(slots, d, k, ws.copies.template as<const void>(),
                                 ws.scale(), ws.nonfinite(), sizes, sums, s, skip);
  };
  if constexpr (std::is_same<T, float>::value) {
    if (ws.tiled) {
      const float *xr = ws.xr.template as<const float>();
      timer.begin(s);
      if (ws.mixed_terms > 0) {
        launch_tiled_mixed_prep(d, k, ws.mixed_terms, cur,
                                ws.hn.template as<const T>(),
                                ws.aop.template as<void>(),
                                ws.bound.template as<float>(), s);
        const bool cand = ws.qmask.bytes() > 0;
        launch_tiled_mixed_assign<I>(n, d, k, ws.mixed_terms, ws.blocks_b, X,
                                     ws.aop.template as<const void>(),
                                     ws.bound.template as<const float>(), labels,
                                     ws.queue.template as<int>(),
                                     ws.queue_counts.template as<int>(),
                                     cand ? ws.qmask.template as<unsigned>() : nullptr,
                                     s, skip, ws.xb.template as<const void>(),
                                     ws.xnb.template as<const float>());
        if (cand)
          launch_tiled_cand_rescore<I>(
              n, d, k, xr, cur, ws.hn.template as<const T>(), labels,
              ws.queue.template as<const int>(),
              ws.queue_counts.template as<const int>(),
              ws.qmask.template as<const unsigned>(), ws.blocks_b, ws.seg_cap,
              ws.cand.template as<void>(), ws.queue_count(), s, skip);
        else
          launch_tiled_rescore<I>(n, d, k, xr, cur, ws.hn.template as<const T>(),
                                  labels, ws.queue.template as<const int>(),
                                  ws.queue_counts.template as<const int>(),
                                  ws.blocks_b, ws.seg_cap, ws.queue_count(), s, skip);
      } else {
        launch_tiled_assign<I>(n, d, k, X, cur, ws.hn.template as<const T>(),
                               labels, s, skip);
      }
      launch_tiled_update<I>(n, d, k, xr, w, labels, ws.scale(),
                             ws.upd.template as<void>(),
                             ws.copies.template as<void>(), s, skip);
      timer.end(s);
      reduce_fixed(1);
      return;
    }
    if (ws.mixed_terms > 0) {
      launch_mixed_prep(d, k, ws.mixed_terms, cur, ws.hn.template as<const T>(),
                        ws.aop.template as<void>(), ws.bound.template as<float>(),
                        s);
      timer.begin(s);
      mixed_labels_and_partials(ws, X, w, cur, labels, s, skip);
      timer.end(s);
      reduce_fixed(ws.blocks + ws.blocks_b);
      return;
    }
  }
  if (ws.fast) {
    timer.begin(s);
    launch_fast_fused_fixed<T, I>(n, d, k, X, w, cur,
                                  ws.hn.template as<const T>(), labels,
                                  ws.scale(), ws.nonfinite(),
                                  ws.copies.template as<void>(), ws.blocks, s, skip);
    timer.end(s);
    reduce_fixed(ws.blocks);
    return;
  }
  if (!ws.store_flush || n == 0) {
    KMD_HIP_CHECK(hipMemsetAsync(ws.copies.template as<T>(), 0,
                                 ws.copies.bytes(), s));
    KMD_HIP_CHECK(hipMemsetAsync(ws.sizes_copies.template as<T>(), 0,
                                 ws.sizes_copies.bytes(), s));
  }
  timer.begin(s);
  if constexpr (std::is_same<T, float>::value) {
    if (ws.wide) {
      launch_wide_assign<I>(n, d, k, X, cur, ws.hn.template as<const T>(), labels, s,
                            skip);
      launch_label_sums<I>(n, d, k, ws.blocks, X, w, cur, labels,
                           ws.copies.template as<T>(),
                           ws.sizes_copies.template as<T>(), s, skip);
    }
  }
  if (!ws.wide)
    launch_fused_generic<T, I>(n, d, k, ws.blocks, ws.plan, ws.store_flush, X,
                               w, cur, ws.hn.template as<const T>(), labels,
                               ws.copies.template as<T>(),
                               ws.sizes_copies.template as<T>(), s, skip);
  timer.end(s);
  launch_sum_copies<T>(ws.blocks, d, k, ws.sizes_copies.template as<const T>(),
                       ws.copies.template as<const T>(), sizes, sums, s, skip);
}

template <typename T, typename I>
static void driver_impl(int64_t n, int64_t d, int64_t k, const T *X, const T *w,
                        T *init, I *labels, T *res, double tol, bool verbose,
                        int64_t max_iter, int64_t *n_iters_out,
                        double *inertia_out, kmd_print_fn print_fn,
                        void *print_user, hipStream_t s, int precision,
                        DriverStats *stats);

template <typename T, typename I>
void driver_lloyd(int64_t n, int64_t d, int64_t k, const T *X, const T *w,
                  T *init, I *labels, T *res, double tol, bool verbose,
                  int64_t max_iter, int64_t *n_iters_out, double *inertia_out,
                  kmd_print_fn print_fn, void *print_user, hipStream_t s,
                  int precision, DriverStats *stats) {
  TuneGuard g(choose_tuning(n, d, k, precision, std::is_same<T, float>::value));
  driver_impl<T, I>(n, d, k, X, w, init, labels, res, tol, verbose, max_iter,
                    n_iters_out, inertia_out, print_fn, print_user, s, precision,
                    stats);
}

// Times the driver's candidate launch plans for this problem and records the
// fastest for its (d, k, precision, log2 n).  Candidates: LDS-resident or
// tiled centroids (where each serves the shape) x persistent blocks per CU
// {occupancy limit, 1, 2, 4}; each runs `iters` Lloyd iterations from the
// given init on scratch copies, timed by the fused step's HIP events (as fits
// of separate launches, also where one block would do the whole fit).  The
// choice never changes results (every plan computes the same labels and
// exact sums).
template <typename T, typename I>
std::vector<TuneResult> autotune_lloyd(int64_t n, int64_t d, int64_t k,
                                       const T *X, const T *w, const T *init,
                                       int precision, int iters, hipStream_t s) {
  std::vector<TuneResult> out;
  if (n <= 0) return out;
  struct Separate {
    Separate() { t_separate = true; }
    ~Separate() { t_separate = false; }
  } separate;
  std::vector<int> paths;
  if (fast_fused_supported<T>(d, k)) paths.push_back(1);
  if (std::is_same<T, float>::value && tiled_supported(d, k)) paths.push_back(2);
  if (paths.empty()) paths.push_back(0);
  TempBuffer c0(sizeof(T) * d * k, s), c1(sizeof(T) * d * k, s),
      lab(sizeof(I) * n, s);
  struct Cand {
    int path, cap, shape;
  };
  std::vector<Cand> cands;
  for (int path : paths) {
    // launch shapes (waves per block x column blocks per wave) of the
    // LDS-resident fixed-point step, then blocks per CU
    const int n_shapes = (path == 1 && std::is_same<T, float>::value) ? 3 : 1;
    for (int shape = 0; shape < n_shapes; ++shape)
      for (int cap : {0, 1, 2, 4}) cands.push_back(Cand{path, cap, shape});
  }
  for (const Cand &cd : cands) {
    {
      const int path = cd.path, cap = cd.cap, shape = cd.shape;
      KMD_HIP_CHECK(hipMemcpyAsync(c0.as<T>(), init, sizeof(T) * d * k,
                                   hipMemcpyDeviceToDevice, s));
      TuneGuard g(TuneChoice{path, cap, shape});
      DriverStats st;
      int64_t it = 0;
      double inertia = 0.0;
      driver_impl<T, I>(n, d, k, X, w, c0.as<T>(), lab.as<I>(), c1.as<T>(), 0.0,
                        false, iters, &it, &inertia, nullptr, nullptr, s,
                        precision, &st);
      TuneResult r;
      r.path = path;
      r.blocks_per_cu = cap;
      r.shape = shape;
      r.ms = st.fused_launches > 0 ? st.fused_kernel_ms / st.fused_launches : 0.0;
      out.push_back(r);
    }
  }
  const TuneResult *best = &out[0];
  for (const TuneResult &r : out)
    if (r.ms > 0.0 && (best->ms <= 0.0 || r.ms < best->ms)) best = &r;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tune[std::make_tuple(d, k, precision, log2_bucket(n))] =
        TuneChoice{best->path, best->blocks_per_cu, best->shape};
  }
  KMD_HIP_CHECK(hipStreamSynchronize(s));
  return out;
}

template <typename T, typename I>
static void driver_impl(int64_t n, int64_t d, int64_t k, const T *X, const T *w,
                        T *init, I *labels, T *res, double tol, bool verbose,
                        int64_t max_iter, int64_t *n_iters_out,
                        double *inertia_out, kmd_print_fn print_fn,
                        void *print_user, hipStream_t s, int precision,
                        DriverStats *stats) {
  auto ws_ptr = make_workspace<T, I>(n, d, k, X, w, precision, s);
  FusedTimer timer(stats != nullptr);
  auto &ws = *ws_ptr;
  // centroid buffers: iteration i reads bufs[i % 2] and writes the other one
  // (when it finds empty clusters: only ws.sums)
  T *bufs[2] = {init, res};
  const T tol_t = static_cast<T>(tol);
  int64_t it = 0;         // iterations known to have finished
  int64_t queued = 0;     // iterations enqueued
  PinnedScalars pinned;
  DrainOnThrow drain{s};
  LoopHost *host = pinned.host();
  // no iteration at all where the sum of shifts could not exceed tol
  if (!(std::numeric_limits<T>::infinity() > tol_t)) max_iter = 0;
  StepTail<T, I> tail{};
  tail.d = d;
  tail.k = k;
  tail.sums = ws.sums.template as<const T>();
  tail.sizes = ws.sizes.template as<const T>();
  tail.shifts = ws.shifts.template as<T>();
  tail.hn = ws.hn.template as<T>();
  tail.list = ws.list.template as<I>();
  tail.state = ws.state();
  tail.host = host;
  tail.rescored = ws.mixed_terms > 0 ? ws.queue_count() : nullptr;
  tail.tol = tol_t;
  tail.partials = ws.tail_part.template as<double>();
  tail.ticket = ws.tail_ticket.template as<unsigned>();
  auto enqueue_tail = [&](int64_t i, bool relocated) {
    tail.cur = bufs[i % 2];
    tail.next = bufs[(i + 1) % 2];
    tail.relocated = relocated ? 1 : 0;
    launch_step_tail<T, I>(tail, s);
  };
  // verbose mode prints between iterations: nothing is enqueued ahead there
  const int ahead = verbose ? 0 : t_run_ahead;
  const bool resident = std::is_same<T, float>::value && ws.fast &&
                        ws.mixed_terms == 0 && !ws.tiled;
  auto finish = [&](double total, int64_t rescored) {
    *inertia_out = static_cast<double>(static_cast<T>(total));
    *n_iters_out = it;
    if (stats) {
      stats->fused_kernel_ms = timer.total_ms;
      stats->fused_launches = timer.launches;
      int path = ws.mixed_terms > 0 ? (ws.mixed_terms == 3 ? 3 : 2)
                                    : (ws.fast ? 1 : 0);
      if (ws.tiled) path += 3;  // 4 tiled FP32, 5 tiled BF16, 6 tiled BF16x3
      if (ws.tiled && ws.mixed_terms == 8) path = 7;  // tiled FP8
      stats->fused_path = path;
      stats->n_rescored = rescored;
    }
  };
  auto start = [&] {   // fixed-point scales (X and w stay as they are), half norms
    if constexpr (std::is_same<T, float>::value) {
      if (resident)
        launch_fixed_point_scales(n, d, X, w, ws.scale(), ws.nonfinite(), s,
                                  ws.stats.template as<void>());
    }
    launch_half_l2_norm<T>(d, k, init, ws.hn.template as<T>(), s);
  };
  // small fits: everything in one launch (up to a relocation)
  bool one_block = resident && !verbose && !t_separate && small_loop_serves(n, d, k);
  if (!one_block) start();
  while (it < max_iter || one_block) {
    if constexpr (std::is_same<T, float>::value) {
      if (one_block) {
        SmallLoop<I> sl{};
        sl.n = n;
        sl.d = (int)d;
        sl.k = (int)k;
        sl.iters = max_iter - it;
        sl.X = X;
        sl.w = w;
        sl.bufs[0] = bufs[0];
        sl.bufs[1] = bufs[1];
        sl.labels = labels;
        sl.sums = ws.sums.template as<float>();
        sl.sizes = ws.sizes.template as<float>();
        sl.per_sample = ws.per_sample.template as<float>();
        sl.list = ws.list.template as<I>();
        sl.state = ws.state();
        sl.host = host;
        sl.tol = tol_t;
        launch_small_loop<I>(sl, s);
      }
    }
    while (!one_block && queued < max_iter && queued <= it + ahead) {
      timer.slot = (int)(queued % (kAhead + 1));
      lloyd_front<T, I>(ws, X, w, bufs[queued % 2], labels, s, timer);
      enqueue_tail(queued, false);
      ++queued;
    }
    const unsigned long long word = wait_loop(host, it, s);
    const int64_t done = (int64_t)(word >> 2);
    int stop = (int)(word & 3);
    if (stop == kLoopRefused) {   // the inputs' range: an iteration per launch
      KMD_HIP_CHECK(hipStreamSynchronize(s));
      KMD_HIP_CHECK(hipMemsetAsync(ws.state(), 0, sizeof(LoopState), s));
      host->word = 0;
      one_block = false;
      start();
      continue;
    }
    if (one_block) {   // no fused step to time
      it = done;
      if (stop == kLoopConverged) {
        KMD_HIP_CHECK(hipStreamSynchronize(s));
        finish(host->total, 0);
        return;
      }
    }
    for (; it < done; ++it) timer.collect((int)(it % (kAhead + 1)));
    T *cur = bufs[(it + 1) % 2];   // of iteration it - 1, the last finished
    if (verbose) {
      launch_inertia<T, I>(n, d, k, X, w, cur, labels,
                           ws.per_sample.template as<T>(), s);
      double tot = 0.0;
      TempBuffer dres(sizeof(double), s);
      launch_reduce_sum<T>(n, ws.per_sample.template as<const T>(),
                           dres.as<double>(), s);
      KMD_HIP_CHECK(hipMemcpyAsync(&tot, dres.as<double>(), sizeof(double),
                                   hipMemcpyDeviceToHost, s));
      KMD_HIP_CHECK(hipStreamSynchronize(s));
      std::ostringstream ss;
      ss << "Iteration: " << it - 1 << " Inertia: " << static_cast<T>(tot);
      if (print_fn) print_fn(ss.str().c_str(), print_user);
    }
    if (stop == kLoopEmpty) {
      // squared distance to the nearest centroid (unit weights), then move
      // the farthest samples into the empty clusters, on the undivided sums;
      // the iterations enqueued ahead skip themselves
      launch_inertia<T, I>(n, d, k, X, nullptr, cur, labels,
                           ws.per_sample.template as<T>(), s);
      launch_relocate<T, I>(n, d, k, host->n_empty, X, w, labels,
                            ws.list.template as<const I>(),
                            ws.per_sample.template as<const T>(),
                            ws.sums.template as<T>(), ws.sizes.template as<T>(),
                            ws.per_sample.template as<T>(), s);
      enqueue_tail(it - 1, true);
      KMD_HIP_CHECK(hipStreamSynchronize(s));
      queued = it;
      stop = (int)(host->word & 3);
    }
    if (stop == kLoopConverged) break;
  }
  // ws.hn holds the half norms of the final centroids: the last tail's, or
  // (no iteration) those of init
  T *cur = bufs[it % 2];

  // epilogue: labels and weighted inertia of the final centroids (on the
  // tiled mixed path with its BF16 kernel and exact re-score: the FP32
  // labels)
  bool labelled = false;
  if constexpr (std::is_same<T, float>::value) {
    if (ws.tiled && ws.mixed_terms > 0 && n > 0) {
      const float *xr = ws.xr.template as<const float>();
      launch_tiled_mixed_prep(d, k, ws.mixed_terms, cur, ws.hn.template as<const T>(),
                              ws.aop.template as<void>(),
                              ws.bound.template as<float>(), s);
      const bool cand = ws.qmask.bytes() > 0;
      launch_tiled_mixed_assign<I>(n, d, k, ws.mixed_terms, ws.blocks_b, X,
                                   ws.aop.template as<const void>(),
                                   ws.bound.template as<const float>(), labels,
                                   ws.queue.template as<int>(),
                                   ws.queue_counts.template as<int>(),
                                   cand ? ws.qmask.template as<unsigned>() : nullptr,
                                   s, nullptr, ws.xb.template as<const void>(),
                                   ws.xnb.template as<const float>());
      if (cand)
        launch_tiled_cand_rescore<I>(
            n, d, k, xr, cur, ws.hn.template as<const T>(), labels,
            ws.queue.template as<const int>(),
            ws.queue_counts.template as<const int>(),
            ws.qmask.template as<const unsigned>(), ws.blocks_b, ws.seg_cap,
            ws.cand.template as<void>(), ws.queue_count(), s);
      else
        launch_tiled_rescore<I>(n, d, k, xr, cur, ws.hn.template as<const T>(),
                                labels, ws.queue.template as<const int>(),
                                ws.queue_counts.template as<const int>(),
                                ws.blocks_b, ws.seg_cap, ws.queue_count(), s);
      labelled = true;
    } else if (ws.mixed_terms > 0 && n > 0) {
      // the BF16 step and its exact re-score: the FP32 labels (its sums go
      // to the partial slots unread)
      launch_mixed_prep(d, k, ws.mixed_terms, cur, ws.hn.template as<const T>(),
                        ws.aop.template as<void>(), ws.bound.template as<float>(),
                        s);
      mixed_labels_and_partials(ws, X, w, cur, labels, s, nullptr);
      labelled = true;
    }
  }
  if (!labelled)
    launch_assignment<T, I>(n, d, k, 0, X, cur, ws.hn.template as<const T>(),
                            labels, s);
  launch_inertia<T, I>(n, d, k, X, w, cur, labels,
                       ws.per_sample.template as<T>(), s);
  if (cur != res)
    KMD_HIP_CHECK(hipMemcpyAsync(res, cur, sizeof(T) * d * k,
                                 hipMemcpyDeviceToDevice, s));
  launch_reduce_sum<T>(n, ws.per_sample.template as<const T>(),
                       ws.epilogue_sum(), s);
  char end[64];   // the loop's state and the epilogue's sum
  KMD_HIP_CHECK(hipMemcpyAsync(end, ws.scalars.template as<char>(), sizeof(end),
                               hipMemcpyDeviceToHost, s));
  KMD_HIP_CHECK(hipStreamSynchronize(s));
  LoopState final_state;
  std::memcpy(&final_state, end, sizeof(final_state));
  double total;
  std::memcpy(&total, end + 56, sizeof(total));
  finish(total, final_state.rescored);
}

#define KMD_INST_DRIVER(T, I)                                                 \
  template void driver_lloyd<T, I>(int64_t, int64_t, int64_t, const T *,     \
                                   const T *, T *, I *, T *, double, bool,    \
                                   int64_t, int64_t *, double *,              \
                                   kmd_print_fn, void *, hipStream_t, int,    \
                                   DriverStats *);                            \
  template std::vector<TuneResult> autotune_lloyd<T, I>(                     \
      int64_t, int64_t, int64_t, const T *, const T *, const T *, int, int,   \
      hipStream_t);
KMD_INST_DRIVER(float, int32_t)
KMD_INST_DRIVER(float, int64_t)
KMD_INST_DRIVER(double, int32_t)
KMD_INST_DRIVER(double, int64_t)

void driver_lloyd_single(const BatchedFit &f, hipStream_t s) {
  driver_lloyd<float, int32_t>(f.n, f.d, f.k, f.X, f.w, f.init, f.labels, f.res,
                               f.tol, false, f.max_iter, f.out_iters,
                               f.out_inertia, nullptr, nullptr, s, KMD_PREC_FP32,
                               nullptr);
}

}  // namespace kmd
