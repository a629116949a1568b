// Float32 shapes beyond the tiled kernels (more than 128 features, or more
// than 32768 clusters): matrix-core labels with the features streamed, and
// the exact centroid sums of given labels.
#include <algorithm>

#include "fixed_point.hpp"
#include "lloyd_fast.hpp"

namespace kmd {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned long long u64;

// ---- labels ------------------------------------------------------------------
//
// A wave owns 32 S samples (columns of v_mfma_f32_32x32x2f32) and keeps the
// accumulators of NT 32-centroid tiles at once, walking the features in
// chunks of kChunkF: a sample's row is then read once per NT tiles however
// long it is, where the tiled kernels (lloyd_tiled.hip) hold it whole in
// registers.  The chunk's centroid rows are staged in LDS for the block's
// four waves, double-buffered; X_t rows come straight from global memory, 32
// consecutive samples per half-wave load, one chunk ahead.  No working
// memory: the centroids are read from the caller's array.
//
// Arithmetic: the chains start from 0 and the score is hn - acc, the order of
// the generic kernel (lloyd.hip); a chain of FP32 MFMAs rounds like fmaf over
// ascending features, so the labels are that kernel's bit for bit.
//
// Bound by the FP32 matrix core: n = 200,003, d = 300, k = 100 takes 0.165 ms
// (the generic kernel: 0.549) where the products alone, 128 columns after
// padding, need 0.100 ms at the 153 TFLOP/s of a large FP32 product; n =
// 400,000, d = 512, k = 512 runs at 115 TFLOP/s.  Measured on the way: address
// arithmetic and bounds masks in vector registers cost a third (0.25 ms), 32
// features per chunk 12 % more than 16.
constexpr int kWNT = 256;
constexpr int kWWaves = kWNT / kWave;
constexpr int kChunkF = 16;             // features per chunk
constexpr int kChunkKs = kChunkF / 2;   // MFMA k-steps per chunk
constexpr int kMaxTiles = 8;

// Word 3 of a raw buffer descriptor on gfx9-family devices (untyped dword
// access, no swizzle).
constexpr int kRsrcWord3 = 0x00020000;

struct WideArgs {
  int64_t n;
  int d, k;
  const float *X, *C, *hn;
  void *labels;
  const int *skip;   // when non-null and *skip != 0 the launch does nothing
};

template <int NT, int S, typename I>
__global__ void __launch_bounds__(kWNT, 2) wide_fp32_krn(WideArgs a) {
  // an iteration enqueued ahead of a relocation: nothing to compute
  if (a.skip != nullptr && *a.skip != 0) return;
  constexpr int KP = 32 * NT;   // centroids of one group of tiles
  constexpr int kPer = kChunkF * KP / kWNT;
  // [4 k-steps][half][centroid][k-step % 4]: a lane's A operands of four
  // k-steps of a tile are one 16-byte read
  __shared__ __align__(16) float Cs[2][kChunkF * KP];
  __shared__ float Hs[KP];                // half norms, +inf padded
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int col = lane & 31, half = lane >> 5;
  const int64_t n = a.n;
  const int d = a.d, k = a.k;
  // All loads go through buffer descriptors that end with what exists, so
  // rows past the last feature, padded centroids and samples past the last
  // one read 0 without a vector instruction: on this chip FP32 products and
  // vector work do not overlap on a SIMD, and address arithmetic and masks
  // would cost a third of the products' time.
  const int64_t s_first = ((int64_t)blockIdx.x * kWWaves + wave) * (32 * S);
  const int64_t s0 = min<int64_t>(s_first, n - 1);
  const int cols = (int)min<int64_t>(32 * S, n - s0);
  // this lane's byte offset from (row f, sample s0): row f + half
  const int xoff = (half ? (int)((unsigned)n * 4u) : 0) + col * 4;
  const int n_chunks = (d + kChunkF - 1) / kChunkF;

  float bestv[S];
  int besti[S];
#pragma unroll
  for (int q = 0; q < S; ++q) {
    bestv[q] = __builtin_huge_valf();
    besti[q] = 0;
  }
  for (int c0 = 0; c0 < k; c0 += KP) {
    float cr[kPer], xn[kChunkKs][S], xr[kChunkKs][S];
    // byte offsets of this thread's elements of a chunk of centroid rows
    int coff[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int e = tid + i * kWNT;
      const int f = e / KP, c = e % KP;
      coff[i] = c0 + c < k ? (f * k + c) * 4 : -4;   // -4: past every end
    }
    auto load_c = [&](int ch) {
      const int f0 = ch * kChunkF;
      const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float *>(a.C + (int64_t)f0 * k + c0), (short)0,
          (min(kChunkF, d - f0) * k - c0) * 4, kRsrcWord3);
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        cr[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, coff[i], 0, 0));
    };
    // rows f and f + 1 (the two halves' rows) of every k-step
    auto load_x = [&](int ch) {
#pragma unroll
      for (int j = 0; j < kChunkKs; ++j) {
        const int f = ch * kChunkF + 2 * j;
        const unsigned last = f + 1 < d ? (unsigned)n + cols : f < d ? cols : 0;
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(a.X + (int64_t)min(f, d - 1) * n + s0), (short)0,
            (int)(last * 4u), kRsrcWord3);
#pragma unroll
        for (int q = 0; q < S; ++q)
          xn[j][q] = __uint_as_float(
              __builtin_amdgcn_raw_buffer_load_b32(r, xoff + 128 * q, 0, 0));
      }
    };
    auto store_c = [&](int buf) {
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int e = tid + i * kWNT;
        const int f = e / KP, c = e % KP;
        Cs[buf][(((f >> 3) * 2 + (f & 1)) * KP + c) * 4 + ((f >> 1) & 3)] = cr[i];
      }
    };
    f32x16 acc[NT][S];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int q = 0; q < S; ++q) acc[t][q] = f32x16{};
    load_c(0);
    load_x(0);
    __syncthreads();   // the previous group's last chunk and half norms are read
    store_c(0);
    for (int c = tid; c < KP; c += kWNT)
      Hs[c] = c0 + c < k ? a.hn[c0 + c] : __builtin_huge_valf();
    __syncthreads();
    for (int ch = 0; ch < n_chunks; ++ch) {
#pragma unroll
      for (int j = 0; j < kChunkKs; ++j)
#pragma unroll
        for (int q = 0; q < S; ++q) xr[j][q] = xn[j][q];
      if (ch + 1 < n_chunks) {
        load_c(ch + 1);
        load_x(ch + 1);
      }
      // items (4 k-steps, tile); the operands are read two items ahead of
      // their products, or every pair of products would wait on LDS
      const float *A = Cs[ch & 1] + (half * KP + col) * 4;
      constexpr int kItems = kChunkKs / 4 * NT;
      auto operands = [&](int i) {
        return *reinterpret_cast<const f32x4 *>(A + ((i / NT) * 2 * KP + 32 * (i % NT)) * 4);
      };
      f32x4 av[3];
      av[0] = operands(0);
      av[1] = operands(kItems > 1 ? 1 : 0);
#pragma unroll
      for (int i = 0; i < kItems; ++i) {
        if (i + 2 < kItems) av[(i + 2) % 3] = operands(i + 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
          for (int q = 0; q < S; ++q)
            acc[i % NT][q] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                av[i % 3][j], xr[4 * (i / NT) + j][q], acc[i % NT][q], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // the other buffer's chunk was last read before the previous barrier
      if (ch + 1 < n_chunks) {
        store_c((ch + 1) & 1);
        __syncthreads();
      }
    }
    // rows of this lane in tile t: 32 t + 8 (r / 4) + 4 half + r % 4, ascending
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = 32 * t + 8 * (r >> 2) + 4 * half + (r & 3);
        const float h = Hs[m];
#pragma unroll
        for (int q = 0; q < S; ++q) {
          const float v = h - acc[t][q][r];
          const bool upd = v < bestv[q];
          bestv[q] = upd ? v : bestv[q];
          besti[q] = upd ? c0 + m : besti[q];
        }
      }
      asm volatile("" ::: "memory");   // one tile's half norms at a time
    }
  }
  // merge the two halves of the column: ties go to the lower centroid
#pragma unroll
  for (int q = 0; q < S; ++q) {
    const float ov = __shfl_xor(bestv[q], 32, kWave);
    const int oi = __shfl_xor(besti[q], 32, kWave);
    if ((ov < bestv[q]) || (ov == bestv[q] && oi < besti[q])) besti[q] = oi;
    const int64_t s = s_first + 32 * q + col;
    if (half == 0 && s < n) reinterpret_cast<I *>(a.labels)[s] = (I)besti[q];
  }
}

using WideFn = void (*)(WideArgs);

// Tiles per group: the groups of about equal size, at most 8 tiles (128
// accumulator registers, two waves per SIMD).  Two column blocks per wave
// halve the LDS reads per product (n = 1,000,000, d = 200, k = 128: 0.464
// against 0.510 ms) where the registers allow it (NT <= 4) and n still gives
// every CU eight blocks (at n = 200,003 the two are equal, at n = 50,000 one
// block is 5 % faster).
template <typename I>
WideFn pick_wide(int nt, bool two) {
  switch (nt) {
    case 1: return two ? &wide_fp32_krn<1, 2, I> : &wide_fp32_krn<1, 1, I>;
    case 2: return two ? &wide_fp32_krn<2, 2, I> : &wide_fp32_krn<2, 1, I>;
    case 3: return two ? &wide_fp32_krn<3, 2, I> : &wide_fp32_krn<3, 1, I>;
    case 4: return two ? &wide_fp32_krn<4, 2, I> : &wide_fp32_krn<4, 1, I>;
    case 5: return &wide_fp32_krn<5, 1, I>;
    case 6: return &wide_fp32_krn<6, 1, I>;
    case 7: return &wide_fp32_krn<7, 1, I>;
    default: return &wide_fp32_krn<8, 1, I>;
  }
}

// ---- sums of given labels ------------------------------------------------------
//
// Block (b, g) adds w_s x_{f,s} over samples [b chunk, (b + 1) chunk) for the
// rows f of group g (row d: the weights) into sums in LDS and the totals, with
// FP32 atomics, into private copy b % n_copies (the accumulate-into contract
// of the fused step).  X_t is read once, coalesced, in the caller's layout;
// labels and weights once per group.
//
// The sums in LDS are the exact int64 binade windows of fixed_point.hpp: no
// pass over X for scales, any input (values outside a window go to the copy
// one by one).  FP32 sums in LDS were measured first: ds_add_f32 took 0.42 ms
// at n = 200,003, d = 300, k = 100; the integer form takes
// 0.072 ms (the read of X alone: 0.051 ms).
constexpr int kSNT = 1024;
constexpr int kSWaves = kSNT / kWave;
constexpr size_t kSumLds = 152 * 1024;   // one block per CU: the fewest totals
constexpr int kSumStep = 8;              // row loads in flight per thread

// exponent of a finite value, 0 of an infinity or NaN
__device__ inline int finite_binade(float v) {
  const int e = (int)((__float_as_uint(v) >> 23) & 0xffu);
  return e != 0xff ? e : 0;
}

template <bool COPIES, typename I>
__global__ void __launch_bounds__(kSNT)
    label_sums_krn(int64_t n, int d, int k, int rows, int rshift, int64_t chunk, int W,
                   const float *__restrict__ X, const float *__restrict__ w,
                   const float *__restrict__ C, const I *__restrict__ labels,
                   float *copies, float *sizes_copies, int n_copies, const int *skip) {
  if (skip != nullptr && *skip != 0) return;
  // [rows][k][1 << rshift] sums, then the rows' windows (whole steps)
  extern __shared__ u64 acc[];
  int *low = reinterpret_cast<int *>(acc + (((int64_t)rows * k) << rshift));
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int f0 = blockIdx.y * rows;
  const int nf = min(rows, d + 1 - f0);   // rows of this group
  const int nx = min(nf, d - f0);         // those of them that are features
  const int64_t beg = blockIdx.x * chunk, s1 = min(n, beg + chunk);
  // The window of feature f ends kWinMargin binades above the largest finite
  // of its centroid coordinates and of the block's first 64 products w x (1 where
  // all of them are 0): of centred data with few clusters the coordinates alone can
  // be far smaller, and then every value went to the copy by itself (n = 200,000,
  // d = 129, k = 2: 2.2 ms instead of 0.04).  That of the weights likewise.
  const int64_t sl = beg + lane;
  const float w0 = sl < s1 ? w[sl] : 0.f;
  constexpr int kRound = 10;   // rows a wave reads side by side (one after another: 2 us each)
  float x[kRound], c[kRound];
  auto load = [&](int fb) {
#pragma unroll
    for (int u = 0; u < kRound; ++u) {
      const int f = fb + u * kSWaves;
      x[u] = f < nx && sl < s1 ? X[(int64_t)(f0 + f) * n + sl] : 1.f;
      c[u] = f < nx && lane < k ? C[(int64_t)(f0 + f) * k + lane] : 0.f;
    }
  };
  load(wave);
  for (int i = threadIdx.x; i < (nf * k) << rshift; i += kSNT) acc[i] = 0ull;
  for (int fb = wave; fb < nf + kSumStep; fb += kRound * kSWaves) {
    if (fb != wave) load(fb);
#pragma unroll
    for (int u = 0; u < kRound; ++u) {
      const int f = fb + u * kSWaves;
      int e = max(finite_binade(x[u] * w0), finite_binade(c[u]));
      if (f < nx)
        for (int cc = kWave + lane; cc < k; cc += kWave)
          e = max(e, finite_binade(C[(int64_t)(f0 + f) * k + cc]));
      for (int o = kWave / 2; o > 0; o >>= 1) e = max(e, __shfl_xor(e, o, kWave));
      if (lane == 0 && f < nf + kSumStep && f < ((rows + kSumStep - 1) & -kSumStep))
        low[f] = window_low(e != 0 ? e : 127, kWinMargin, W);
    }
  }
  __syncthreads();
  const int64_t copy = blockIdx.x % (unsigned)n_copies;
  float *out = copies + (copy * d + f0) * k;
  float *out_w = sizes_copies + copy * k;
  const int own = lane & ((1 << rshift) - 1);
  for (int64_t s = beg + threadIdx.x; s < s1; s += kSNT) {
    const int l = (int)labels[s];
    const float ws = w[s];
    const float *col = X + (int64_t)f0 * n + s;
    auto add = [&](int f, float v) {
      const int off = f * k + l;
      window_add(acc + (COPIES ? (off << rshift) + own : off), out + off, 0, v, low[f], W);
    };
    int f = 0;
    for (; f + kSumStep <= nx; f += kSumStep) {
      float x[kSumStep];
#pragma unroll
      for (int j = 0; j < kSumStep; ++j) x[j] = col[(int64_t)(f + j) * n];
#pragma unroll
      for (int j = 0; j < kSumStep; ++j) add(f + j, x[j] * ws);
    }
    if (f < nx) {   // (a product of 0 is added nowhere)
      float x[kSumStep];
#pragma unroll
      for (int j = 0; j < kSumStep; ++j) x[j] = f + j < nx ? col[(int64_t)(f + j) * n] : 0.f;
#pragma unroll
      for (int j = 0; j < kSumStep; ++j) add(f + j, f + j < nx ? x[j] * ws : 0.f);
    }
    if (nx < nf) {
      const int off = nx * k + l;
      window_add(acc + (COPIES ? (off << rshift) + own : off), out_w + l, 0, ws, low[nx], W);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nf * k; i += kSNT) {
    const int f = i / k;
    u64 t = 0;
    for (int r = 0; r < 1 << rshift; ++r) t += acc[(i << rshift) + ((r + lane) & ((1 << rshift) - 1))];
    const float v = (float)ldexp((double)(long long)t, low[f] - 150);
    if (v != 0.f) atomic_add(f < nx ? out + i : out_w + (i - nx * k), v);
  }
}

struct SumPlan {
  int rows, rshift;
  int64_t groups, blocks;   // of rows; of samples
};

inline size_t sum_lds(int64_t rows, int64_t k, int rshift) {
  return (sizeof(u64) * (size_t)k << rshift) * rows +
         sizeof(int) * (ceil_div<int64_t>(rows, kSumStep) * kSumStep);
}

// Groups of rows: as few as LDS allows, of about equal size, for labels and weights
// are read once per group; with few samples more of them, so that the blocks are
// near one per CU (never more: four blocks past that are a second round of all),
// a block taking at least 2048 samples.
//
// Copies of a sum: lanes of one label add to one address, one after the other, so
// the lanes of a wave have 64 sums of a row or more between them.
//
// A fused step with one sum each and groups as few as LDS allows, whatever n, against
// this: n = 3000, d = 800, k = 8: 907 -> 85 us; n = 40,000, d = 128, k = 2: 257 -> 105;
// n = 10,000, d = 400, k = 20: 338 -> 84.
SumPlan plan_sums(int64_t n, int64_t d, int64_t k) {
  SumPlan p{};
  while ((k << p.rshift) < kWave && p.rshift < 5) ++p.rshift;
  int64_t most = std::max<int64_t>(1, (int64_t)kSumLds / (int64_t)(sizeof(u64) * k << p.rshift));
  while (most > 1 && sum_lds(most, k, p.rshift) > kSumLds) --most;
  const int64_t cus = device_cu_count();
  p.groups = ceil_div<int64_t>(d + 1, most);
  p.blocks = std::max<int64_t>(1, std::min<int64_t>(cus / p.groups, ceil_div<int64_t>(n, 2048)));
  p.rows = (int)ceil_div<int64_t>(d + 1, p.groups);
  if (cus / p.blocks > p.groups) {
    const int64_t r = ceil_div<int64_t>(d + 1, cus / p.blocks);
    p.rows = (int)std::min<int64_t>(p.rows, ceil_div<int64_t>(r, kSumStep) * kSumStep);
    p.groups = ceil_div<int64_t>(d + 1, p.rows);
  }
  return p;
}

}  // namespace

bool wide_supported(int64_t n, int64_t d, int64_t k) {
  // 32-bit element offsets inside a pair of sample rows and inside a chunk
  // of centroid rows
  return n >= 1 && n < (int64_t(1) << 29) && d >= 1 && d < (int64_t(1) << 30) &&
         k >= 1 && k < (int64_t(1) << 25);
}

template <typename I>
void launch_wide_assign(int64_t n, int64_t d, int64_t k, const float *X_t,
                        const float *C, const float *hn, I *labels,
                        hipStream_t s, const int *skip) {
  if (n <= 0) return;
  WideArgs a{};
  a.n = n;
  a.d = (int)d;
  a.k = (int)k;
  a.X = X_t;
  a.C = C;
  a.hn = hn;
  a.labels = labels;
  a.skip = skip;
  require(wide_supported(n, d, k), "wide assignment: unsupported shape");
  const int n_ct = (int)ceil_div<int64_t>(k, 32);
  const int nt = ceil_div(n_ct, ceil_div(n_ct, kMaxTiles));
  const bool two = nt <= 4 && n >= 8 * (int64_t)device_cu_count() * 64 * kWWaves;
  hipLaunchKernelGGL(pick_wide<I>(nt, two),
                     dim3((unsigned)ceil_div<int64_t>(n, (two ? 64 : 32) * kWWaves)),
                     dim3(kWNT), 0, s, a);
  KMD_LAUNCH_CHECK();
}

// one row of sums fits kSumLds
bool label_sums_supported(int64_t k) {
  return k >= 1 && (size_t)k * sizeof(u64) + sizeof(int) <= kSumLds;   // (and a few windows)
}

// label_update_krn's sums are 4 bytes, so it holds twice the rows; the 8 bytes a
// sum here have to be cleared and flushed for the samples to pay for.  Steps of d
// = 16 to 128, this against that one: k <= 1024 0.81 - 1.02 x at any n; n >= 8 k up
// to the k whose rows stand two at a time in LDS 0.83 - 1.02 x; n = 2 k there 1.00 -
// 1.05 x; one row at a time (n = 1M, d = 128, k = 10,000) 1272 us against 780.
bool label_sums_first(int64_t n, int64_t k) {
  return label_sums_supported(k) &&
         sum_lds(2, k, 0) <= kSumLds && (k <= 1024 || n >= 8 * k);
}

template <typename I>
void launch_label_sums(int64_t n, int64_t d, int64_t k, int64_t n_copies,
                       const float *X_t, const float *w, const float *C,
                       const I *labels, float *copies, float *sizes_copies,
                       hipStream_t s, const int *skip) {
  if (n <= 0) return;
  require(label_sums_supported(k), "label sums: too many clusters for one LDS row");
  const SumPlan p = plan_sums(n, d, k);
  const int64_t chunk = ceil_div<int64_t>(n, p.blocks);
  auto fn = p.rshift > 0 ? &label_sums_krn<true, I> : &label_sums_krn<false, I>;
  allow_full_lds(reinterpret_cast<const void *>(fn));
  hipLaunchKernelGGL(fn, dim3((unsigned)p.blocks, (unsigned)p.groups),
                     dim3(kSNT), sum_lds(p.rows, k, p.rshift), s, n, (int)d, (int)k, p.rows,
                     p.rshift, chunk, window_width(chunk), X_t, w, C, labels, copies,
                     sizes_copies, (int)n_copies, skip);
  KMD_LAUNCH_CHECK();
}

#define KMD_INST_WIDE(I)                                                      \
  template void launch_wide_assign<I>(int64_t, int64_t, int64_t, const float *, \
                                      const float *, const float *, I *,      \
                                      hipStream_t, const int *);              \
  template void launch_label_sums<I>(int64_t, int64_t, int64_t, int64_t,      \
                                     const float *, const float *,            \
                                     const float *, const I *, float *,       \
                                     float *, hipStream_t, const int *);
KMD_INST_WIDE(int32_t)
KMD_INST_WIDE(int64_t)

}  // namespace kmd
