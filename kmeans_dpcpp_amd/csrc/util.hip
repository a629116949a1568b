// Small wave-level kernels around the Lloyd step: broadcast divide, half
// squared norms, private-copy reduction with the empty-cluster list, centroid
// shifts, per-sample inertia, deterministic sum / max reductions, selection of
// far samples and empty-cluster relocation.
#include <algorithm>

#include "common.hpp"
#include "lloyd_fast.hpp"

namespace kmd {

namespace {

constexpr int kBlock = 256;

__device__ inline int lane_id() { return threadIdx.x & (kWave - 1); }

// Block-wide sum of a double (256 threads); result valid in every thread.
__device__ inline double block_sum(double v, double *lds /*[kBlock/kWave]*/) {
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  const int w = threadIdx.x / kWave;
  __syncthreads();
  if (lane_id() == 0) lds[w] = v;
  __syncthreads();
  double t = 0.0;
  for (int i = 0; i < (int)(blockDim.x / kWave); ++i) t += lds[i];
  return t;
}

// ---- broadcast divide: x[r, c] /= y[c] (src/util_kernels.hpp:9-41) ---------
template <typename T>
__global__ void __launch_bounds__(kBlock)
    broadcast_divide_krn(int64_t total, int64_t n_cols, T *x, const T *y) {
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * kBlock) {
    x[i] = x[i] / y[i % n_cols];
  }
}

// ---- half squared norms (src/util_kernels.hpp:47-82) -----------------------
// Column c, rows ascending, fused multiply-add accumulation, then / 2.  The
// chain of a column is serial, so its values are staged in LDS by the whole
// block first: 32 columns x 64 rows at a time, all loads in flight.  One
// thread per column reading global memory took 69 us at d = 300, k = 100
// (each of the d dependent steps waits on L2), this form 15 us in a cold cache.
constexpr int kHnCols = 32, kHnRows = 64;

template <typename T>
__global__ void __launch_bounds__(kBlock)
    half_l2_norm_krn(int64_t d, int64_t k, const T *__restrict__ C, T *__restrict__ out) {
  __shared__ T v[kHnRows][kHnCols + 1];
  const int e = threadIdx.x % kHnCols, g = threadIdx.x / kHnCols;
  const int64_t c = blockIdx.x * (int64_t)kHnCols + e;
  T acc = T(0);
  for (int64_t f0 = 0; f0 < d; f0 += kHnRows) {
    __syncthreads();
#pragma unroll
    for (int r = g; r < kHnRows; r += kBlock / kHnCols)
      v[r][e] = (f0 + r < d && c < k) ? C[(f0 + r) * k + c] : T(0);
    __syncthreads();
    const int m = (int)min<int64_t>(kHnRows, d - f0);
    if (g == 0)
      for (int r = 0; r < m; ++r) acc = fma(v[r][e], v[r][e], acc);
  }
  if (g == 0 && c < k) out[c] = acc / T(2);
}

// ---- reduce private copies (src/util_kernels.hpp:84-161) -------------------
// Elements i < dk: centroid sums, out_cent[i] = sum over copies of
// cent[copy * dk + i]; the k after them: cluster sizes.  A 1024-thread block
// owns 1024 / G consecutive elements; its thread groups each sum the copies
// congruent to their index mod G (ascending), then the G partial sums are
// added in ascending order: a fixed order, so the result is deterministic.
// Few elements in many copies (few clusters: 264 elements in 695 copies)
// leave most of the chip idle with G = 16; G = 64 gives four times the blocks
// and a quarter of the serial additions (35 us in two launches before, 9 us
// in one).
constexpr int kRedThreads = 1024;
constexpr int kRedElems = 64;
constexpr int kRedGroups = 16;

template <typename T, int G>
__global__ void __launch_bounds__(kRedThreads)
    sum_copies_krn(int64_t n_copies, int64_t dk, int64_t k, const T *__restrict__ cent,
                   const T *__restrict__ sizes, T *__restrict__ out_cent,
                   T *__restrict__ out_sizes, const int *skip) {
  if (skip != nullptr && *skip != 0) return;
  constexpr int E = kRedThreads / G;
  __shared__ T part[G][E + 1];
  const int e = threadIdx.x % E, g = threadIdx.x / E;
  const int64_t i = blockIdx.x * (int64_t)E + e;
  const bool is_cent = i < dk;
  const T *src = is_cent ? cent + i : sizes + (i - dk);
  const int64_t stride = is_cent ? dk : k;
  T acc = T(0);
  if (i < dk + k) {
    int64_t c = g;
    for (; c + 3 * G < n_copies; c += 4 * G) {
      const T a0 = src[c * stride];
      const T a1 = src[(c + G) * stride];
      const T a2 = src[(c + 2 * G) * stride];
      const T a3 = src[(c + 3 * G) * stride];
      acc += a0;
      acc += a1;
      acc += a2;
      acc += a3;
    }
    for (; c < n_copies; c += G) acc += src[c * stride];
  }
  part[g][e] = acc;
  __syncthreads();
  if (g == 0 && i < dk + k) {
    T t = T(0);
    for (int q = 0; q < G; ++q) t += part[q][e];
    (is_cent ? out_cent[i] : out_sizes[i - dk]) = t;
  }
}

// Per-block partials of the MFMA fused step, [n_blocks][d*k + k]: int64
// fixed-point sums (exact, so any summation order gives the same result),
// converted once with the feature's scale; or FP32 sums in a fixed order
// when the inputs held non-finite values.
template <typename T>
__global__ void __launch_bounds__(kRedThreads)
    sum_partials_fixed_krn(int64_t n_blocks, int64_t d, int64_t k,
                           const void *__restrict__ partials,
                           const float *__restrict__ scale,
                           const int *__restrict__ nonfinite,
                           T *__restrict__ out_sizes, T *__restrict__ out_cent,
                           const int *skip) {
  if (skip != nullptr && *skip != 0) return;
  __shared__ long long ipart[kRedGroups][kRedElems];
  __shared__ float fpart[kRedGroups][kRedElems];
  const int e = threadIdx.x % kRedElems, g = threadIdx.x / kRedElems;
  const int64_t m = d * k + k;
  const int64_t i = blockIdx.x * (int64_t)kRedElems + e;
  const bool fixed = nonfinite[0] == 0;
  long long iacc = 0;
  float facc = 0.f;
  if (i < m) {
    if (fixed) {
      const long long *p = reinterpret_cast<const long long *>(partials);
      for (int64_t c = g; c < n_blocks; c += kRedGroups) iacc += p[c * m + i];
    } else {
      const float *p = reinterpret_cast<const float *>(partials);
      for (int64_t c = g; c < n_blocks; c += kRedGroups) facc += p[c * m + i];
    }
  }
  ipart[g][e] = iacc;
  fpart[g][e] = facc;
  __syncthreads();
  if (g == 0 && i < m) {
    T v;
    if (fixed) {
      long long t = 0;
      for (int q = 0; q < kRedGroups; ++q) t += ipart[q][e];
      const int64_t f = i / k;  // == d for the counts
      v = (T)((double)t / (double)scale[f]);
    } else {
      float t = 0.f;
      for (int q = 0; q < kRedGroups; ++q) t += fpart[q][e];
      v = (T)t;
    }
    if (i < d * k)
      out_cent[i] = v;
    else
      out_sizes[i - d * k] = v;
  }
}

// Appends every cluster with size 0 to empty_list at n_empty[0]++, in
// ascending cluster order (one block; prefix sums over ballots).
template <typename T, typename I>
__global__ void __launch_bounds__(1024)
    empty_list_krn(int64_t k, const T *__restrict__ sizes, I *empty_list,
                   I *n_empty, int64_t list_len) {
  __shared__ int wave_counts[1024 / kWave];
  __shared__ int64_t running;
  if (threadIdx.x == 0) running = (int64_t)n_empty[0];
  __syncthreads();
  const int nwaves = blockDim.x / kWave;
  const int w = threadIdx.x / kWave;
  for (int64_t c0 = 0; c0 < k; c0 += blockDim.x) {
    const int64_t c = c0 + threadIdx.x;
    const bool empty = (c < k) && (sizes[c] == T(0));
    const uint64_t mask = __ballot(empty);
    const int before_in_wave = __popcll(mask & ((1ull << lane_id()) - 1ull));
    if (lane_id() == 0) wave_counts[w] = __popcll(mask);
    __syncthreads();
    int before = 0, total = 0;
    for (int i = 0; i < nwaves; ++i) {
      before += (i < w) ? wave_counts[i] : 0;
      total += wave_counts[i];
    }
    if (empty) {
      const int64_t pos = running + before + before_in_wave;
      if (pos >= 0 && pos < list_len) empty_list[pos] = (I)c;
    }
    __syncthreads();
    if (threadIdx.x == 0) running += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) n_empty[0] = (I)running;
}

// ---- centroid shifts (src/util_kernels.hpp:478-516) ------------------------
template <typename T>
__global__ void __launch_bounds__(kBlock)
    centroid_shifts_krn(int64_t d, int64_t k, const T *a, const T *b, T *out) {
  int64_t c = blockIdx.x * (int64_t)kBlock + threadIdx.x;
  if (c >= k) return;
  T acc = T(0);
  for (int64_t f = 0; f < d; ++f) {
    T diff = a[f * k + c] - b[f * k + c];
    acc = fma(diff, diff, acc);
  }
  out[c] = acc;
}

// ---- end of a Lloyd iteration ------------------------------------------------
// From the undivided sums and sizes: the empty-cluster list, or (no cluster
// empty) next = sums / sizes (src/util_kernels.hpp:9-41), shift[c] = sum_f
// (cur - next)^2 in feature order (src/util_kernels.hpp:478-516), the half
// norms of the new centroids as half_l2_norm_krn computes them, the FP64 sum
// of the shifts, and the loop's state on the device and in host memory.  A
// finished loop (stop != 0: converged, or clusters to relocate) makes the
// kernels enqueued after it return at once.
//
// Column tiles are staged in LDS by the whole block (all loads in flight)
// before the serial chains over the features; a thread per column reading
// global memory, and a launch for the list, took 38 + 5 us at d = 300, k =
// 100 and 5.4 + 2.7 us at d = 14, k = 127, where this takes 16 and 4.7 us.
// Shapes that fit one tile (d = 32, k = 256 does) run on one block and keep
// the shifts in registers (65 us for one block over six tiles, d = 96, k =
// 512: 17 us with the others); the others run a block per tile, at most
// kTailBlocks (the ticket's atomics serialise), and the last one to finish
// adds up the shifts.
constexpr int kTailThreads = 1024;
constexpr int kTailValues = 8192;        // values of one LDS tile
constexpr int kTailSmall = 2048;         // wanted values of one of many tiles
constexpr int kTailBlocks = 64;

// Columns of one tile: a power of two up to kTailThreads.
inline int tail_cols(int64_t d, int64_t k) {
  auto pow2_up = [](int64_t v) {
    int64_t p = 1;
    while (p < v) p *= 2;
    return p;
  };
  const int64_t whole = pow2_up(k);
  if (whole <= kTailThreads && d * whole <= kTailValues) return (int)whole;
  int64_t ct = 8;
  while (2 * ct * d <= kTailSmall) ct *= 2;
  ct = std::max(ct, pow2_up(ceil_div<int64_t>(k, kTailBlocks)));
  return (int)std::min<int64_t>(ct, kTailThreads);
}

template <typename T, typename I>
__global__ void __launch_bounds__(kTailThreads)
    step_tail_krn(StepTail<T, I> a, int CT) {
  extern __shared__ __align__(16) unsigned char tail_smem[];
  T *qv = reinterpret_cast<T *>(tail_smem);   // [rows][CT] new centroids
  T *cv = qv + kTailValues;                   // [rows][CT] old centroids
  double *lds = reinterpret_cast<double *>(cv + kTailValues);   // one per wave
  int *wave_counts = reinterpret_cast<int *>(lds + kTailThreads / kWave);
  int &last = wave_counts[kTailThreads / kWave];
  const int tid = threadIdx.x, wave = tid / kWave;
  const int64_t d = a.d, k = a.k;
  if (!a.relocated) {
    // Whether the loop has stopped is read by one thread, so that a block goes
    // on or returns as one: with clusters empty, block 0 sets `stop` as soon as
    // it has listed them, while blocks that start later still read it.  Both
    // answers end such a block (a stopped loop, or its own look at the sizes),
    // and no block of that launch takes a ticket.
    if (tid == 0)
      last = __hip_atomic_load(&a.state->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // every block looks for empty clusters itself; block 0 lists them
    bool any = tid < k && a.sizes[tid] == T(0);
    for (int64_t c = tid + kTailThreads; c < k; c += kTailThreads)
      any |= a.sizes[c] == T(0);
    const uint64_t any_mask = __ballot(any);
    if (lane_id() == 0) wave_counts[wave] = any_mask != 0;
    __syncthreads();
    if (last != 0) return;
    int n_any = 0;
    for (int i = 0; i < kTailThreads / kWave; ++i) n_any += wave_counts[i];
    if (n_any != 0) {
      if (blockIdx.x != 0) return;
      int64_t found = 0;
      for (int64_t c0 = 0; c0 < k; c0 += kTailThreads) {
        const int64_t c = c0 + tid;
        const bool empty = c < k && a.sizes[c] == T(0);
        const uint64_t mask = __ballot(empty);
        __syncthreads();
        if (lane_id() == 0) wave_counts[wave] = __popcll(mask);
        __syncthreads();
        int before = 0, total = 0;
        for (int i = 0; i < kTailThreads / kWave; ++i) {
          before += i < wave ? wave_counts[i] : 0;
          total += wave_counts[i];
        }
        if (empty)
          a.list[found + before + __popcll(mask & ((1ull << lane_id()) - 1ull))] = (I)c;
        found += total;
      }
      if (tid == 0) {
        LoopState *st = a.state;
        st->n_empty = found;
        st->rescored += a.rescored != nullptr ? a.rescored[0] : 0;
        st->done += 1;
        __hip_atomic_store(&st->stop, kLoopEmpty, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        publish(a.host, *st);
      }
      return;
    }
  }

  const int rows = kTailValues / CT;
  const int e = tid & (CT - 1);              // this thread's column of a tile
  const int r0 = tid / CT, rstep = kTailThreads / CT;
  const int64_t n_tiles = (k + CT - 1) / CT;
  T acc = T(0);
  for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const int64_t c0 = tile * CT;
    const int64_t c = c0 + tid;
    const bool col = c0 + e < k;
    const T size = col ? a.sizes[c0 + e] : T(1);
    T h = T(0);
    acc = T(0);
    for (int64_t f0 = 0; f0 < d; f0 += rows) {
      const int m = (int)min<int64_t>(rows, d - f0);
      __syncthreads();
      constexpr int kU = 4;   // rows loaded ahead of their use
      for (int r = r0; r < m; r += kU * rstep) {
        T sv[kU], ov[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int64_t at = (f0 + r + u * rstep) * k + c0 + e;
          const bool in = col && r + u * rstep < m;
          sv[u] = in ? a.sums[at] : T(0);
          ov[u] = in ? a.cur[at] : T(0);
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int64_t at = (f0 + r + u * rstep) * k + c0 + e;
          if (col && r + u * rstep < m) {
            const T q = sv[u] / size;
            a.next[at] = q;
            qv[(r + u * rstep) * CT + e] = q;
            cv[(r + u * rstep) * CT + e] = ov[u];
          }
        }
      }
      __syncthreads();
      if (tid < CT && c < k) {
#pragma unroll 8
        for (int r = 0; r < m; ++r) {
          const T q = qv[r * CT + tid], diff = cv[r * CT + tid] - q;
          acc = fma(diff, diff, acc);
          h = fma(q, q, h);
        }
      }
    }
    if (tid < CT && c < k) {
      a.hn[c] = h / T(2);
      if (n_tiles > 1) a.shifts[c] = acc;
    }
  }
  // Sum of the shifts in FP64: the 64 columns of a wave by exchanges, the four
  // waves of each 256 columns, then those sums by 256 threads the same way.
  auto wave_sum = [](double v) {
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
  };
  double tot = 0.0;
  if (n_tiles == 1) {   // k <= 1024: at most four sums of 256 columns
    const double t = wave_sum(tid < k ? (double)acc : 0.0);
    if (lane_id() == 0) lds[wave] = t;
    __syncthreads();
    if (tid != 0) return;
    double p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      p[j] = 0.0;
      for (int i = 0; i < 4; ++i) p[j] += lds[4 * j + i];
    }
    tot = (p[0] + p[2]) + (p[1] + p[3]);   // the exchanges' order
  } else {
    if (gridDim.x > 1) {
      __threadfence();
      __syncthreads();
      if (tid == 0) last = atomicAdd(a.ticket, 1u) == gridDim.x - 1 ? 1 : 0;
      __syncthreads();
      if (last == 0) return;
      __threadfence();
    } else {
      __syncthreads();
    }
    for (int64_t c0 = 0; c0 < k; c0 += kTailThreads) {
      const int64_t c = c0 + tid;
      const double v =
          c < k ? (double)__hip_atomic_load(&a.shifts[c], __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT)
                : 0.0;
      const double t = wave_sum(v);
      __syncthreads();
      if (lane_id() == 0) lds[wave] = t;
      __syncthreads();
      if (tid < kTailThreads / 256 && c0 + 256 * tid < k) {
        double u = 0.0;
        for (int i = 0; i < 4; ++i) u += lds[4 * tid + i];
        a.partials[c0 / 256 + tid] = u;
      }
    }
    __syncthreads();
    const int64_t nb = (k + 255) / 256;
    double v = 0.0;
    if (tid < 256)
      for (int64_t i = tid; i < nb; i += 256) v += a.partials[i];
    const double t = wave_sum(v);
    if (lane_id() == 0) lds[wave] = t;
    __syncthreads();
    if (tid != 0) return;
    for (int i = 0; i < 4; ++i) tot += lds[i];
    if (gridDim.x > 1) a.ticket[0] = 0u;
  }
  LoopState *st = a.state;
  st->shift = tot;
  if (!a.relocated) {
    st->rescored += a.rescored != nullptr ? a.rescored[0] : 0;
    st->done += 1;
  }
  // the loop goes on while the sum, in the data type, exceeds tol
  st->stop = (T)tot > a.tol ? 0 : kLoopConverged;
  publish(a.host, *st);
}

// ---- per-sample inertia (src/compute_inertia.hpp:11-99) --------------------
template <typename T, typename I>
__global__ void __launch_bounds__(kBlock)
    inertia_krn(int64_t n, int64_t d, int64_t k, const T *X, const T *w,
                const T *C, const I *labels, T *out) {
  for (int64_t s = blockIdx.x * (int64_t)kBlock + threadIdx.x; s < n;
       s += (int64_t)gridDim.x * kBlock) {
    int64_t c = (int64_t)labels[s];
    T acc = T(0);
    if (c >= 0 && c < k) {
      for (int64_t f = 0; f < d; ++f) {
        T diff = X[f * n + s] - C[f * k + c];
        acc = fma(diff, diff, acc);
      }
    } else {
      acc = std::numeric_limits<T>::quiet_NaN();
    }
    out[s] = (w != nullptr) ? acc * w[s] : acc;
  }
}

// The same with the centroids staged in LDS as k rows of d + 1 values (row
// c = centroid c; the odd stride puts lanes with different c mod 32 on
// different banks), for k (d + 1) values within kInertiaLds bytes: each
// sample's d centroid reads come from LDS instead of a 64-address gather per
// wave load.  Same arithmetic and order per sample as inertia_krn.
constexpr size_t kInertiaLds = 64 * 1024;
template <typename T, typename I>
__global__ void __launch_bounds__(kBlock)
    inertia_lds_krn(int64_t n, int64_t d, int64_t k, const T *X, const T *w,
                    const T *C, const I *labels, T *out) {
  extern __shared__ __align__(16) unsigned char inertia_smem[];
  T *Cs = reinterpret_cast<T *>(inertia_smem);
  const int64_t ld = d + 1;
  for (int64_t e = threadIdx.x; e < d * k; e += kBlock) {
    const int64_t f = e / k, c = e - f * k;
    Cs[c * ld + f] = C[e];
  }
  __syncthreads();
  for (int64_t s = blockIdx.x * (int64_t)kBlock + threadIdx.x; s < n;
       s += (int64_t)gridDim.x * kBlock) {
    int64_t c = (int64_t)labels[s];
    T acc = T(0);
    if (c >= 0 && c < k) {
      // up to kU feature loads in flight (one round for d <= kU); the fma
      // chain still runs over f = 0, 1, ...
      constexpr int kU = 32;
      const T *row = Cs + c * ld;
      for (int64_t f0 = 0; f0 < d; f0 += kU) {
        T xv[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) xv[u] = (f0 + u < d) ? X[(f0 + u) * n + s] : T(0);
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          if (f0 + u < d) {
            T diff = xv[u] - row[f0 + u];
            acc = fma(diff, diff, acc);
          }
        }
      }
    } else {
      acc = std::numeric_limits<T>::quiet_NaN();
    }
    out[s] = (w != nullptr) ? acc * w[s] : acc;
  }
}

// The same for centroids beyond kInertiaLds: kF features of all centroids at a
// time in LDS (feature-major rows as they are in memory), the chains of P samples
// a thread in registers meanwhile.  A gather of C[f][labels] from L2 touches up to
// 64 lines per wave load and bounds inertia_krn (n = 2M, d = 128, k = 1024: 594
// us); here the gather is an LDS read and X's own pass is what is left (239 us,
// 4.3 TB/s).  Each tile of 1024 P samples stages all of C and few tiles leave the
// chip idle, so the rule asks for n >= kInertiaRatio k: at n = 64 k the gather is
// the faster one (n = 65,536, d = 128, k = 1024, double: 65 us against 53 or
// less), at 250 k and 16 features both take the same (67 us), at 488 k and 64
// features 181 us against 73 (double: 334 against 134).
constexpr int kInertiaThreads = 1024;
constexpr int64_t kInertiaRatio = 256;
template <int kF, int P, typename T, typename I>
__global__ void __launch_bounds__(kInertiaThreads)
    inertia_chunk_krn(int64_t n, int d, int k, const T *__restrict__ X,
                      const T *__restrict__ w, const T *__restrict__ C,
                      const I *__restrict__ labels, T *out) {
  extern __shared__ __align__(16) unsigned char inertia_smem[];
  T *Cs = reinterpret_cast<T *>(inertia_smem);
  constexpr int kTile = kInertiaThreads * P;
  for (int64_t s0 = blockIdx.x * (int64_t)kTile; s0 < n; s0 += (int64_t)gridDim.x * kTile) {
    int64_t at[P];
    int c[P];
    T acc[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int64_t s = s0 + p * kInertiaThreads + threadIdx.x;
      at[p] = s < n ? s : n - 1;
      const int64_t l = (int64_t)labels[at[p]];
      acc[p] = (l >= 0 && l < k) ? T(0) : std::numeric_limits<T>::quiet_NaN();
      c[p] = (l >= 0 && l < k) ? (int)l : 0;
    }
    for (int f0 = 0; f0 < d; f0 += kF) {
      const int nf = min(kF, d - f0);
      T xv[P][kF];
#pragma unroll
      for (int u = 0; u < kF; ++u)
#pragma unroll
        for (int p = 0; p < P; ++p)
          xv[p][u] = u < nf ? X[(int64_t)(f0 + u) * n + at[p]] : T(0);
      __syncthreads();
      for (int e = threadIdx.x; e < nf * k; e += kInertiaThreads)
        Cs[e] = C[(int64_t)f0 * k + e];
      __syncthreads();
#pragma unroll
      for (int u = 0; u < kF; ++u) {
        if (u < nf) {
#pragma unroll
          for (int p = 0; p < P; ++p) {
            const T diff = xv[p][u] - Cs[u * k + c[p]];
            acc[p] = fma(diff, diff, acc[p]);
          }
        }
      }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int64_t s = s0 + p * kInertiaThreads + threadIdx.x;
      if (s < n) out[s] = (w != nullptr) ? acc[p] * w[s] : acc[p];
    }
  }
}

// ---- deterministic two-stage sum (src/compute_inertia.hpp:104-135) ---------
// Stage 1: fixed grid, each block sums a grid-stride slice in FP64.
template <typename T>
__global__ void __launch_bounds__(kBlock)
    sum_stage1_krn(int64_t n, const T *x, double *partials) {
  __shared__ double lds[kBlock / kWave];
  double acc = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock)
    acc += (double)x[i];
  double t = block_sum(acc, lds);
  if (threadIdx.x == 0) partials[blockIdx.x] = t;
}

template <typename OutT>
__global__ void __launch_bounds__(kBlock)
    sum_stage2_krn(int nb, const double *partials, OutT *out) {
  __shared__ double lds[kBlock / kWave];
  double acc = 0.0;
  for (int i = threadIdx.x; i < nb; i += kBlock) acc += partials[i];
  double t = block_sum(acc, lds);
  if (threadIdx.x == 0) out[0] = (OutT)t;
}

// ---- max reduction (src/util_kernels.hpp:174-188); NaN is ignored ----------
template <typename T>
__global__ void __launch_bounds__(kBlock)
    max_stage_krn(int64_t n, const T *x, T *out) {
  __shared__ T lds[kBlock / kWave];
  T m = -std::numeric_limits<T>::infinity();
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock) {
    T v = x[i];
    m = (v > m) ? v : m;
  }
  for (int o = kWave / 2; o > 0; o >>= 1) {
    T v = __shfl_xor(m, o, kWave);
    m = (v > m) ? v : m;
  }
  if (lane_id() == 0) lds[threadIdx.x / kWave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    T r = lds[0];
    for (int i = 1; i < kBlock / kWave; ++i) r = (lds[i] > r) ? lds[i] : r;
    out[blockIdx.x] = r;
  }
}

// ---- select samples far from centroids (src/util_kernels.hpp:208-297) -----
// Deterministic stable compaction in three launches: per-block counts,
// scatter, counter update.  Each block owns a contiguous chunk.
template <typename T>
__global__ void __launch_bounds__(kBlock)
    select_count_krn(int64_t n, int64_t chunk, const T *dist, const T *thr,
                     int64_t *counts /*[2*nb]*/) {
  __shared__ int64_t lds[2][kBlock / kWave];
  const T t = thr[0];
  int64_t lo = blockIdx.x * chunk, hi = min(n, lo + chunk);
  int64_t gt = 0, eq = 0;
  for (int64_t i = lo + threadIdx.x; i < hi; i += kBlock) {
    T v = dist[i];
    gt += (v > t);
    eq += (v == t);
  }
  for (int o = kWave / 2; o > 0; o >>= 1) {
    gt += __shfl_xor(gt, o, kWave);
    eq += __shfl_xor(eq, o, kWave);
  }
  if (lane_id() == 0) {
    lds[0][threadIdx.x / kWave] = gt;
    lds[1][threadIdx.x / kWave] = eq;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t a = 0, b = 0;
    for (int i = 0; i < kBlock / kWave; ++i) {
      a += lds[0][i];
      b += lds[1][i];
    }
    counts[2 * blockIdx.x] = a;
    counts[2 * blockIdx.x + 1] = b;
  }
}

template <typename T, typename I>
__global__ void __launch_bounds__(kBlock)
    select_scatter_krn(int64_t n, int64_t chunk, int64_t n_selected,
                       const T *dist, const T *thr, const int64_t *counts,
                       int nb, I *selected, const I *n_gt, const I *n_eq) {
  __shared__ int64_t off_gt, off_eq, tot_gt;
  __shared__ int wc[2][kBlock / kWave];
  __shared__ int64_t red[3][kBlock / kWave];
  {  // this block's offsets and the total: integer sums over the blocks' counts
    int64_t a = 0, b = 0, ta = 0;
    for (int i = threadIdx.x; i < nb; i += kBlock) {
      const int64_t cg = counts[2 * i], ce = counts[2 * i + 1];
      if (i < (int)blockIdx.x) {
        a += cg;
        b += ce;
      }
      ta += cg;
    }
    for (int o = kWave / 2; o > 0; o >>= 1) {
      a += __shfl_xor(a, o, kWave);
      b += __shfl_xor(b, o, kWave);
      ta += __shfl_xor(ta, o, kWave);
    }
    if (lane_id() == 0) {
      red[0][threadIdx.x / kWave] = a;
      red[1][threadIdx.x / kWave] = b;
      red[2][threadIdx.x / kWave] = ta;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int64_t ra = 0, rb = 0, rt = 0;
      for (int q = 0; q < kBlock / kWave; ++q) {
        ra += red[0][q];
        rb += red[1][q];
        rt += red[2][q];
      }
      off_gt = ra;
      off_eq = rb;
      tot_gt = rt;
    }
  }
  __syncthreads();
  const T t = thr[0];
  const int64_t base_gt = (int64_t)n_gt[0];
  const int64_t base_eq = (int64_t)n_eq[0];
  const int64_t eq_limit = max((int64_t)0, n_selected - tot_gt);
  int64_t run_gt = off_gt, run_eq = off_eq;
  const int w = threadIdx.x / kWave;
  int64_t lo = blockIdx.x * chunk, hi = min(n, lo + chunk);
  for (int64_t i0 = lo; i0 < hi; i0 += kBlock) {
    int64_t i = i0 + threadIdx.x;
    bool g = false, e = false;
    if (i < hi) {
      T v = dist[i];
      g = v > t;
      e = v == t;
    }
    uint64_t mg = __ballot(g), me = __ballot(e);
    uint64_t below = (1ull << lane_id()) - 1ull;
    if (lane_id() == 0) {
      wc[0][w] = __popcll(mg);
      wc[1][w] = __popcll(me);
    }
    __syncthreads();
    int bg = 0, be = 0, tg = 0, te = 0;
    for (int q = 0; q < kBlock / kWave; ++q) {
      bg += (q < w) ? wc[0][q] : 0;
      be += (q < w) ? wc[1][q] : 0;
      tg += wc[0][q];
      te += wc[1][q];
    }
    if (g) {
      int64_t pos = base_gt + run_gt + bg + __popcll(mg & below);
      if (pos >= 0 && pos < n) selected[pos] = (I)i;
    }
    if (e) {
      int64_t r = run_eq + be + __popcll(me & below);
      if (r < eq_limit) {
        int64_t pos = n - (base_eq + r);
        if (pos >= 0 && pos < n) selected[pos] = (I)i;
      }
    }
    run_gt += tg;
    run_eq += te;
    __syncthreads();
  }
}

template <typename I>
__global__ void __launch_bounds__(kBlock)
    select_finalize_krn(int64_t n_selected, const int64_t *counts, int nb, I *n_gt,
                        I *n_eq) {
  __shared__ int64_t red[2][kBlock / kWave];
  int64_t a = 0, b = 0;
  for (int i = threadIdx.x; i < nb; i += kBlock) {
    a += counts[2 * i];
    b += counts[2 * i + 1];
  }
  for (int o = kWave / 2; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, kWave);
    b += __shfl_xor(b, o, kWave);
  }
  if (lane_id() == 0) {
    red[0][threadIdx.x / kWave] = a;
    red[1][threadIdx.x / kWave] = b;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  a = 0;
  b = 0;
  for (int q = 0; q < kBlock / kWave; ++q) {
    a += red[0][q];
    b += red[1][q];
  }
  int64_t eq_limit = n_selected - a;
  if (eq_limit < 0) eq_limit = 0;
  n_gt[0] = (I)((int64_t)n_gt[0] + a);
  n_eq[0] = (I)((int64_t)n_eq[0] + (b < eq_limit ? b : eq_limit));
}

// ---- relocation ordering + application (src/util_kernels.hpp:302-390) -----
// order[j] = j-th farthest sample by (sq_dist desc, index asc), j < m.
// Inputs: selected[0:g] = indices with dist > T (ascending index),
// selected[n-1], selected[n-2], ... = indices with dist == T (ascending).
template <typename T, typename I>
__global__ void __launch_bounds__(1024)
    relocation_order_krn(int64_t n, int64_t m, const T *dist,
                         const I *selected, const I *n_gt, const I *n_eq,
                         int64_t *order) {
  const int64_t g = (int64_t)n_gt[0];
  const int64_t e = (int64_t)n_eq[0] - 1;  // eq counter started at 1
  for (int64_t i = threadIdx.x; i < g; i += blockDim.x) {
    int64_t si = (int64_t)selected[i];
    T di = dist[si];
    int64_t rank = 0;
    for (int64_t j = 0; j < g; ++j) {
      int64_t sj = (int64_t)selected[j];
      T dj = dist[sj];
      rank += (dj > di) || (dj == di && sj < si);
    }
    if (rank < m) order[rank] = si;
  }
  for (int64_t r = threadIdx.x; r < e; r += blockDim.x) {
    int64_t pos = g + r;
    if (pos < m) order[pos] = (int64_t)selected[n - 1 - r];
  }
  // NaN distances can leave fewer samples than m: no sample for the rest
  // (as far_order_krn)
  for (int64_t pos = g + (e > 0 ? e : 0) + threadIdx.x; pos < m; pos += blockDim.x)
    order[pos] = -1;
}

// The same order in one launch of one block, for n <= kFarN samples and m <=
// kFarM of them: thirteen launches of the general way (threshold, selection,
// order) are mostly latency there.  The whole relocation of m = 2 of n = 50,000:
// 237 -> 111 us (this kernel 19), n = 262,144: 253 -> 147 us; one CU reads at 60 -
// 70 GB/s, and past that n the general way's cost stays where it is while this
// one's grows with n.  The m-th largest of the threads' own maxima bounds the
// m-th largest distance from below; the samples above it, about 1.4 m at half as
// many as threads, are gathered in LDS and ranked (m = 200 of 50,000: 331 -> 212
// us).  With m near the number of threads that bound is no bound any more (m =
// 1000 of 50,000: 775 -> 963 us), hence kFarM.  Many equal distances can make the
// list overflow all the same: then the m-th largest is found over all samples,
// and the equal ones are taken in index order.  A NaN distance (key 0) is never
// far: with fewer than m others, the places after them hold no sample (-1).
constexpr int64_t kFarN = 262144;
constexpr int kFarThreads = 1024;
constexpr int64_t kFarM = kFarThreads / 2;
constexpr int kFarList = 2048;

template <typename T>
struct FarKey;
template <>
struct FarKey<float> {
  using U = unsigned;
  static __device__ U of(float v) {
    const U b = __float_as_uint(v + 0.f);   // -0 as +0
    return v != v ? 0u : (b >> 31) ? ~b : (b | 0x80000000u);
  }
};
template <>
struct FarKey<double> {
  using U = unsigned long long;
  static __device__ U of(double v) {
    const U b = (U)__double_as_longlong(v + 0.0);
    return v != v ? 0ull : (b >> 63) ? ~b : (b | (1ull << 63));
  }
};

template <typename T>
__global__ void __launch_bounds__(kFarThreads)
    far_order_krn(int n, int m, const T *__restrict__ dist, int64_t *__restrict__ order) {
  using U = typename FarKey<T>::U;
  constexpr int kWaves = kFarThreads / kWave;
  __shared__ U lkey[kFarList];
  __shared__ int lidx[kFarList];
  __shared__ int wc[2][kWaves];
  __shared__ int count;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  // sum of every wave's v over the block; par alternates between calls
  auto block_count = [&](int v, int par) {
    if (lane == 0) wc[par][wave] = v;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) t += wc[par][i];
    return t;
  };
  if (tid == 0) count = 0;
  U mine = 0;
  constexpr int kU = 8;
  for (int i0 = tid; i0 < n; i0 += kU * kFarThreads) {
    T v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int i = i0 + u * kFarThreads;
      v[u] = i < n ? dist[i] : std::numeric_limits<T>::quiet_NaN();
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const U q = FarKey<T>::of(v[u]);
      mine = q > mine ? q : mine;
    }
  }
  // largest key that at least m of the threads' maxima reach, bit by bit
  U low = 0;
  int par = 0;
  for (int b = 8 * (int)sizeof(U) - 1; b >= 0; --b, par ^= 1) {
    const U probe = low | (U(1) << b);
    if (block_count(__popcll(__ballot(mine >= probe)), par) >= m) low = probe;
  }
  for (int i0 = tid; i0 < n; i0 += kU * kFarThreads) {
    T v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int i = i0 + u * kFarThreads;
      v[u] = i < n ? dist[i] : T(0);
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int i = i0 + u * kFarThreads;
      const U q = FarKey<T>::of(v[u]);
      if (i < n && q != 0 && q >= low) {
        const int at = atomicAdd(&count, 1);
        if (at < kFarList) {
          lkey[at] = q;
          lidx[at] = i;
        }
      }
    }
  }
  __syncthreads();
  int listed = count;
  if (listed > kFarList) {
    // (kFarList > kFarM: at least m samples are no NaN, so thr below is not 0)
    // the exact m-th largest key, then the samples above it and the first
    // ones equal to it
    U thr = 0;
    for (int b = 8 * (int)sizeof(U) - 1; b >= 0; --b, par ^= 1) {
      const U probe = thr | (U(1) << b);
      int c = 0;
      for (int i = tid; i - lane < n; i += kFarThreads)
        c += __popcll(__ballot(i < n && FarKey<T>::of(dist[min(i, n - 1)]) >= probe));
      if (block_count(c, par) >= m) thr = probe;
    }
    __syncthreads();
    if (tid == 0) count = 0;
    __syncthreads();
    for (int i = tid; i < n; i += kFarThreads) {
      const U q = FarKey<T>::of(dist[i]);
      if (q > thr) {
        const int at = atomicAdd(&count, 1);   // fewer than m <= kFarM of them
        lkey[at] = q;
        lidx[at] = i;
      }
    }
    __syncthreads();
    int have = count;
    for (int i0 = 0; i0 < n && have < m; i0 += kFarThreads, par ^= 1) {
      const int i = i0 + tid;
      const bool eq = i < n && FarKey<T>::of(dist[min(i, n - 1)]) == thr;
      const unsigned long long mask = __ballot(eq);
      const int total = block_count(__popcll(mask), par);
      int before = 0;
      for (int q = 0; q < wave; ++q) before += wc[par][q];
      const int at = have + before + __popcll(mask & ((1ull << lane) - 1ull));
      if (eq && at < m) {
        lkey[at] = thr;
        lidx[at] = i;
      }
      have += total;
    }
    __syncthreads();
    listed = min(have, m);
  }
  for (int i = tid; i < listed; i += kFarThreads) {
    const U ki = lkey[i];
    const int si = lidx[i];
    int rank = 0;
    for (int j = 0; j < listed; ++j) {
      const U kj = lkey[j];
      rank += (kj > ki) || (kj == ki && lidx[j] < si);
    }
    if (rank < m) order[rank] = si;
  }
  for (int r = listed + tid; r < m; r += kFarThreads) order[r] = -1;
}

template <typename T, typename I>
__global__ void __launch_bounds__(kBlock)
    relocate_apply_krn(int64_t n, int64_t d, int64_t k, int64_t m,
                       const T *X, const T *w, const I *labels,
                       const I *empty_list, const int64_t *order, T *C,
                       T *sizes, T *inertia) {
  int64_t f = blockIdx.x * (int64_t)kBlock + threadIdx.x;
  if (f >= d) return;
  for (int64_t j = 0; j < m; ++j) {
    int64_t s = order[j];
    int64_t e = (int64_t)empty_list[j];
    const bool none = s < 0 || s >= n;
    int64_t p = (int64_t)labels[none ? 0 : s];
    if (none || p < 0 || p >= k || e < 0 || e >= k) continue;
    T ws = w[s];
    T add = X[f * n + s] * ws;
    C[f * k + p] -= add;
    C[f * k + e] = add;
    if (f == 0) {
      sizes[p] -= ws;
      sizes[e] = ws;
      inertia[s] = T(0);
    }
  }
}

template <typename T, typename I>
__global__ void init_counters_krn(I *n_gt, I *n_eq) {
  n_gt[0] = I(0);
  n_eq[0] = I(1);
}

// The sums of sum_copies_krn, both arrays in one launch.
template <typename T>
void sum_copies(int64_t n_copies, int64_t dk, int64_t k, const T *cent, const T *sizes,
                T *out_cent, T *out_sizes, hipStream_t s, const int *skip) {
  if (dk + k <= 0) return;
  if (n_copies >= 256 && dk + k <= 16384) {
    hipLaunchKernelGGL((sum_copies_krn<T, 64>),
                       dim3((unsigned)ceil_div<int64_t>(dk + k, kRedThreads / 64)),
                       dim3(kRedThreads), 0, s, n_copies, dk, k, cent, sizes, out_cent,
                       out_sizes, skip);
  } else {
    hipLaunchKernelGGL((sum_copies_krn<T, kRedGroups>),
                       dim3((unsigned)ceil_div<int64_t>(dk + k, kRedElems)),
                       dim3(kRedThreads), 0, s, n_copies, dk, k, cent, sizes, out_cent,
                       out_sizes, skip);
  }
  KMD_LAUNCH_CHECK();
}

inline int grid_for(int64_t n, int per_block, int cap) {
  int64_t g = ceil_div<int64_t>(n, per_block);
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (int)g;
}

}  // namespace

// ---- launchers ---------------------------------------------------------------

template <typename T>
void launch_broadcast_divide(int64_t n_rows, int64_t n_cols, T *x, const T *y,
                             hipStream_t s) {
  int64_t total = n_rows * n_cols;
  if (total == 0) return;
  hipLaunchKernelGGL(broadcast_divide_krn<T>, dim3(grid_for(total, kBlock, 65536)),
                     dim3(kBlock), 0, s, total, n_cols, x, y);
  KMD_LAUNCH_CHECK();
}

template <typename T>
void launch_half_l2_norm(int64_t d, int64_t k, const T *C, T *out,
                         hipStream_t s) {
  if (k == 0) return;
  hipLaunchKernelGGL(half_l2_norm_krn<T>, dim3((unsigned)ceil_div<int64_t>(k, kHnCols)),
                     dim3(kBlock), 0, s, d, k, C, out);
  KMD_LAUNCH_CHECK();
}

template <typename T, typename I>
void launch_reduce_centroids(int64_t n_copies, int64_t d, int64_t k,
                             const T *sizes_copies, const T *cent_copies,
                             T *out_sizes, T *out_cent, I *empty_list,
                             I *n_empty, int64_t list_len, hipStream_t s) {
  sum_copies<T>(n_copies, d * k, k, cent_copies, sizes_copies, out_cent, out_sizes, s,
                nullptr);
  hipLaunchKernelGGL((empty_list_krn<T, I>), dim3(1), dim3(1024), 0, s, k,
                     (const T *)out_sizes, empty_list, n_empty, list_len);
  KMD_LAUNCH_CHECK();
}

template <typename T>
void launch_sum_copies(int64_t n_copies, int64_t d, int64_t k, const T *sizes_copies,
                       const T *cent_copies, T *out_sizes, T *out_cent, hipStream_t s,
                       const int *skip) {
  sum_copies<T>(n_copies, d * k, k, cent_copies, sizes_copies, out_cent, out_sizes, s,
                skip);
}

template <typename T>
void launch_sum_fixed_partials(int64_t n_blocks, int64_t d, int64_t k,
                               const void *partials, const float *scale,
                               const int *nonfinite, T *out_sizes, T *out_cent,
                               hipStream_t s, const int *skip) {
  const int64_t m = d * k + k;
  hipLaunchKernelGGL(sum_partials_fixed_krn<T>,
                     dim3((unsigned)ceil_div<int64_t>(m, kRedElems)), dim3(kRedThreads), 0,
                     s, n_blocks, d, k, partials, scale, nonfinite, out_sizes, out_cent,
                     skip);
  KMD_LAUNCH_CHECK();
}

template <typename T>
void launch_centroid_shifts(int64_t d, int64_t k, const T *a, const T *b,
                            T *out, hipStream_t s) {
  if (k == 0) return;
  hipLaunchKernelGGL(centroid_shifts_krn<T>, dim3(ceil_div<int64_t>(k, kBlock)),
                     dim3(kBlock), 0, s, d, k, a, b, out);
  KMD_LAUNCH_CHECK();
}

int64_t step_tail_partials(int64_t k) { return ceil_div<int64_t>(k > 0 ? k : 1, 256); }

template <typename T, typename I>
void launch_step_tail(const StepTail<T, I> &a, hipStream_t s) {
  const int CT = tail_cols(a.d, a.k);
  const unsigned blocks =
      (unsigned)std::min<int64_t>(ceil_div<int64_t>(a.k, CT), kTailBlocks);
  const size_t lds = 2 * sizeof(T) * kTailValues +
                     (kTailThreads / kWave) * (sizeof(double) + sizeof(int)) + sizeof(double);
  allow_full_lds(reinterpret_cast<const void *>(&step_tail_krn<T, I>));
  hipLaunchKernelGGL((step_tail_krn<T, I>), dim3(blocks), dim3(kTailThreads), lds, s, a, CT);
  KMD_LAUNCH_CHECK();
}

template <typename T, typename I>
void launch_inertia(int64_t n, int64_t d, int64_t k, const T *X, const T *w,
                    const T *C, const I *labels, T *out, hipStream_t s) {
  if (n == 0) return;
  const size_t lds = sizeof(T) * (size_t)k * (size_t)(d + 1);
  if (lds <= kInertiaLds) {
    static const bool attr_set = [] {
      KMD_HIP_CHECK(hipFuncSetAttribute(
          reinterpret_cast<const void *>(&inertia_lds_krn<T, I>),
          hipFuncAttributeMaxDynamicSharedMemorySize, (int)kInertiaLds));
      return true;
    }();
    (void)attr_set;
    // persistent blocks, each staging the centroids once: as many per CU as
    // the 160 KB of LDS hold, at most 8 (32 waves)
    const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(8, (160 * 1024) / (int64_t)lds));
    const int64_t grid = std::min<int64_t>(ceil_div<int64_t>(n, kBlock),
                                           (int64_t)device_cu_count() * per_cu);
    hipLaunchKernelGGL((inertia_lds_krn<T, I>), dim3((unsigned)grid), dim3(kBlock), lds, s,
                       n, d, k, X, w, C, labels, out);
    KMD_LAUNCH_CHECK();
    return;
  }
  constexpr int64_t kRow = kInertiaLds / sizeof(T);   // values of C a block stages
  if (4 * k <= kRow && n >= kInertiaRatio * k && d <= INT32_MAX) {
    const bool f8 = 8 * k <= kRow;
    const bool two = n > (int64_t)device_cu_count() * 2 * kInertiaThreads;
    auto fn = f8 ? (two ? inertia_chunk_krn<8, 2, T, I> : inertia_chunk_krn<8, 1, T, I>)
                 : (two ? inertia_chunk_krn<4, 2, T, I> : inertia_chunk_krn<4, 1, T, I>);
    const int64_t tiles = ceil_div<int64_t>(n, kInertiaThreads * (two ? 2 : 1));
    const int64_t grid = std::min<int64_t>(tiles, (int64_t)device_cu_count() * 2);
    hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(kInertiaThreads),
                       sizeof(T) * (size_t)k * (f8 ? 8 : 4), s, n, (int)d, (int)k, X, w, C,
                       labels, out);
    KMD_LAUNCH_CHECK();
    return;
  }
  hipLaunchKernelGGL((inertia_krn<T, I>), dim3(grid_for(n, kBlock, 8192)),
                     dim3(kBlock), 0, s, n, d, k, X, w, C, labels, out);
  KMD_LAUNCH_CHECK();
}

static int sum_blocks(int64_t n) { return grid_for(n, kBlock * 16, 1024); }

template <typename T>
void launch_reduce_sum(int64_t n, const T *x, double *dev_result,
                       hipStream_t s) {
  const int nb = sum_blocks(n);
  TempBuffer partials(sizeof(double) * nb, s);
  hipLaunchKernelGGL(sum_stage1_krn<T>, dim3(nb), dim3(kBlock), 0, s, n, x,
                     partials.as<double>());
  KMD_LAUNCH_CHECK();
  hipLaunchKernelGGL(sum_stage2_krn<double>, dim3(1), dim3(kBlock), 0, s, nb,
                     partials.as<const double>(), dev_result);
  KMD_LAUNCH_CHECK();
}

template <typename T>
void launch_sum_to_scalar(int64_t n, const T *x, T *dev_result,
                          hipStream_t s) {
  const int nb = sum_blocks(n);
  TempBuffer partials(sizeof(double) * nb, s);
  hipLaunchKernelGGL(sum_stage1_krn<T>, dim3(nb), dim3(kBlock), 0, s, n, x,
                     partials.as<double>());
  KMD_LAUNCH_CHECK();
  hipLaunchKernelGGL(sum_stage2_krn<T>, dim3(1), dim3(kBlock), 0, s, nb,
                     partials.as<const double>(), dev_result);
  KMD_LAUNCH_CHECK();
}

template <typename T>
void launch_max(int64_t n, const T *x, T *out, hipStream_t s) {
  const int nb = grid_for(n, kBlock * 16, 1024);
  TempBuffer partials(sizeof(T) * nb, s);
  hipLaunchKernelGGL(max_stage_krn<T>, dim3(nb), dim3(kBlock), 0, s, n, x,
                     partials.as<T>());
  KMD_LAUNCH_CHECK();
  hipLaunchKernelGGL(max_stage_krn<T>, dim3(1), dim3(kBlock), 0, s, (int64_t)nb,
                     partials.as<const T>(), out);
  KMD_LAUNCH_CHECK();
}

template <typename T, typename I>
void launch_select_far(int64_t n_selected, int64_t n, const T *dist,
                       const T *thr, I *selected, I *n_gt, I *n_eq,
                       hipStream_t s) {
  const int nb = grid_for(n, kBlock * 32, 1024);
  const int64_t chunk = ceil_div<int64_t>(n, nb);
  TempBuffer counts(sizeof(int64_t) * 2 * nb, s);
  hipLaunchKernelGGL(select_count_krn<T>, dim3(nb), dim3(kBlock), 0, s, n,
                     chunk, dist, thr, counts.as<int64_t>());
  KMD_LAUNCH_CHECK();
  hipLaunchKernelGGL((select_scatter_krn<T, I>), dim3(nb), dim3(kBlock), 0, s,
                     n, chunk, n_selected, dist, thr,
                     counts.as<const int64_t>(), nb, selected, n_gt, n_eq);
  KMD_LAUNCH_CHECK();
  hipLaunchKernelGGL(select_finalize_krn<I>, dim3(1), dim3(kBlock), 0, s,
                     n_selected, counts.as<const int64_t>(), nb, n_gt, n_eq);
  KMD_LAUNCH_CHECK();
}

template <typename T, typename I>
void launch_relocate(int64_t n, int64_t d, int64_t k, int64_t n_empty,
                     const T *X, const T *w, const I *labels,
                     const I *empty_list, const T *sq_dist, T *centroids,
                     T *sizes, T *per_sample_inertia, hipStream_t s) {
  const int64_t m = n_empty < n ? n_empty : n;
  if (m <= 0 || d <= 0) return;
  TempBuffer order(sizeof(int64_t) * m, s);
  // (released behind the last launch: a release in front of it is a marker in the
  // stream that the launch waits behind, 10 us)
  TempBuffer thr(0, s), sel(0, s);
  if (n <= kFarN && m <= kFarM) {
    hipLaunchKernelGGL(far_order_krn<T>, dim3(1), dim3(kFarThreads), 0, s, (int)n, (int)m,
                       sq_dist, order.as<int64_t>());
    KMD_LAUNCH_CHECK();
  } else {
    thr = TempBuffer(sizeof(T), s);
    sel = TempBuffer(sizeof(I) * (n + 2), s);
    I *n_gt = sel.as<I>() + n;
    I *n_eq = n_gt + 1;
    launch_far_threshold<T>(n, sq_dist, m, thr.as<T>(), s);
    hipLaunchKernelGGL((init_counters_krn<T, I>), dim3(1), dim3(1), 0, s, n_gt, n_eq);
    KMD_LAUNCH_CHECK();
    launch_select_far<T, I>(m, n, sq_dist, thr.as<const T>(), sel.as<I>(), n_gt, n_eq, s);
    hipLaunchKernelGGL((relocation_order_krn<T, I>), dim3(1), dim3(1024), 0, s, n, m,
                       sq_dist, sel.as<const I>(), n_gt, n_eq, order.as<int64_t>());
    KMD_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL((relocate_apply_krn<T, I>), dim3(ceil_div<int64_t>(d, kBlock)),
                     dim3(kBlock), 0, s, n, d, k, m, X, w, labels, empty_list,
                     order.as<const int64_t>(), centroids, sizes,
                     per_sample_inertia);
  KMD_LAUNCH_CHECK();
}

// ---- explicit instantiations -----------------------------------------------
#define KMD_INST_T(T)                                                          \
  template void launch_broadcast_divide<T>(int64_t, int64_t, T *, const T *,  \
                                           hipStream_t);                      \
  template void launch_half_l2_norm<T>(int64_t, int64_t, const T *, T *,      \
                                       hipStream_t);                          \
  template void launch_centroid_shifts<T>(int64_t, int64_t, const T *,        \
                                          const T *, T *, hipStream_t);       \
  template void launch_reduce_sum<T>(int64_t, const T *, double *,            \
                                     hipStream_t);                            \
  template void launch_sum_to_scalar<T>(int64_t, const T *, T *,              \
                                        hipStream_t);                         \
  template void launch_max<T>(int64_t, const T *, T *, hipStream_t);           \
  template void launch_sum_copies<T>(int64_t, int64_t, int64_t, const T *,    \
                                     const T *, T *, T *, hipStream_t,        \
                                     const int *);                            \
  template void launch_sum_fixed_partials<T>(                                 \
      int64_t, int64_t, int64_t, const void *, const float *, const int *,    \
      T *, T *, hipStream_t, const int *);
KMD_INST_T(float)
KMD_INST_T(double)

#define KMD_INST_TI(T, I)                                                     \
  template void launch_reduce_centroids<T, I>(                                \
      int64_t, int64_t, int64_t, const T *, const T *, T *, T *, I *, I *,    \
      int64_t, hipStream_t);                                                  \
  template void launch_inertia<T, I>(int64_t, int64_t, int64_t, const T *,   \
                                     const T *, const T *, const I *, T *,    \
                                     hipStream_t);                            \
  template void launch_select_far<T, I>(int64_t, int64_t, const T *,         \
                                        const T *, I *, I *, I *,             \
                                        hipStream_t);                         \
  template void launch_relocate<T, I>(int64_t, int64_t, int64_t, int64_t,    \
                                      const T *, const T *, const I *,        \
                                      const I *, const T *, T *, T *, T *,    \
                                      hipStream_t);                           \
  template void launch_step_tail<T, I>(const StepTail<T, I> &, hipStream_t);
KMD_INST_TI(float, int32_t)
KMD_INST_TI(float, int64_t)
KMD_INST_TI(double, int32_t)
KMD_INST_TI(double, int64_t)

}  // namespace kmd
