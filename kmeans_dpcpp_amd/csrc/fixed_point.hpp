// Fixed-point scales of the exact centroid sums, shared by the single-fit and
// batched kernels so that both quantise every sample identically.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace kmd {

// Layout of the statistics gathered over X and w before a fit:
//   maxbits[f], f < d : max over samples of (bit pattern of X[f, s]) & 0x7fffffff
//   maxbits[d]        : the same for the weights
//   maxbits[d + 1]    : max over non-zero weights of ~(bits & 0x7fffffff), i.e.
//                       the complement of the smallest non-zero |w| (0: none)
//   estat[2 f], estat[2 f + 1] (f <= d): sum and count of the exponent fields
//                       of the row's normal (non-zero, finite) values
inline constexpr int64_t range_maxbits_count(int64_t d) { return d + 2; }
inline constexpr int64_t range_estat_count(int64_t d) { return 2 * (d + 1); }

// Adds one value's bit pattern to a thread's running maximum and exponent
// sum / count.
__device__ inline void range_accumulate(unsigned bits, unsigned &m, unsigned &esum,
                                        unsigned &ecnt) {
  const unsigned b = bits & 0x7fffffffu;
  m = b > m ? b : m;
  const unsigned e = b >> 23;
  const bool normal = e - 1u < 254u;
  esum += normal ? e : 0u;
  ecnt += normal ? 1u : 0u;
}

// Largest spread, in binary orders of magnitude, between the largest value
// of a row and the geometric mean of its normal values, beyond which the
// fixed-point sums are not used: with the step 2^-30 of the largest
// |w x_f|, a value of typical size keeps at least 30 - 12 = 18 bits.
constexpr double kMaxTypicalSpread = 12.0;
// Largest spread between the largest and the smallest non-zero weight: every
// weight (and so every count) keeps at least 30 - 13 = 17 bits.
constexpr int kMaxWeightSpread = 13;

// scale[f] = 2^E_f with max|w| max|x_f| 2^E_f < 2^30 (each rounded element
// fits an int32) and n max|w| max|x_f| 2^E_f < 2^61 (the sum fits an int64);
// scale[d] likewise for the counts.
// *flag = 1 if any value is infinite or NaN; else 2 if the data's dynamic
// range would leave typical elements (or the smallest weight) coarsely
// quantised (spreads above kMaxTypicalSpread / kMaxWeightSpread; estat may be
// NULL to skip this test); else 0.  Kernels sum in floating point whenever
// *flag != 0.
// The scale of one row whose largest |w x_f| (or |w|) is m.
__device__ inline float fixed_point_scale(int64_t n, double m) {
  int e = 0;
  if (m > 0.0 && m < 1e300) {
    int ex_elem, ex_sum;
    frexp(m, &ex_elem);                       // m < 2^ex_elem
    frexp(m * (double)(n > 0 ? n : 1), &ex_sum);
    const int e1 = 30 - ex_elem, e2 = 61 - ex_sum;
    e = e1 < e2 ? e1 : e2;
    e = e > 120 ? 120 : (e < -120 ? -120 : e);
  }
  return ldexpf(1.f, e);
}

// Binary orders of magnitude from the geometric mean of row f's normal values
// to its largest.
__device__ inline double fixed_point_spread(int f, const unsigned *maxbits,
                                            const unsigned long long *estat) {
  const unsigned long long cnt = estat[2 * f + 1];
  if (cnt == 0) return 0.0;
  const double mean_e = (double)estat[2 * f] / (double)cnt;
  return (double)(maxbits[f] >> 23) - mean_e;
}

// *flag from what the rows gave: bad, any value not finite; sx, the largest
// spread of a feature (estat != NULL).
__device__ inline int fixed_point_flag(int d, bool bad, double sx, const unsigned *maxbits,
                                       const unsigned long long *estat) {
  if (bad) return 1;
  bool coarse = false;
  if (estat != nullptr) {
    coarse |= sx + fixed_point_spread(d, maxbits, estat) > kMaxTypicalSpread;
    const unsigned wmin_inv = maxbits[d + 1];
    if (wmin_inv != 0u) {
      const int emin = (int)((~wmin_inv & 0x7fffffffu) >> 23);
      coarse |= (int)(maxbits[d] >> 23) - emin > kMaxWeightSpread;
    }
  }
  return coarse ? 2 : 0;
}

// One thread.
__device__ inline void fixed_point_scales_from_bits(
    int64_t n, int d, const unsigned *maxbits, const unsigned long long *estat,
    float *scale, int *flag) {
  const unsigned wb = maxbits[d];
  bool bad = wb >= 0x7f800000u;
  const double wmax = (double)__uint_as_float(wb);
  double sx = 0.0;
  for (int f = 0; f <= d; ++f) {
    const unsigned b = maxbits[f];
    bad |= b >= 0x7f800000u;
    scale[f] = fixed_point_scale(n, wmax * (f < d ? (double)__uint_as_float(b) : 1.0));
    if (f < d && estat != nullptr) {
      const double sf = fixed_point_spread(f, maxbits, estat);
      sx = sf > sx ? sf : sx;
    }
  }
  flag[0] = fixed_point_flag(d, bad, sx, maxbits, estat);
}

// Exact binade-window sums (for the steps that run no pass over X for
// scales).  A finite FP32 value v = m 2^(e - 150) (m the
// 24-bit significand, e the biased exponent) whose binade e lies in
// [lo, lo + W] is the integer m << (e - lo) in units of 2^(lo - 150), with
// no rounding: those values go into the block's int64 LDS sums exactly
// (|m << W| < 2^(24 + W) leaves 2^(39 - W) additions of headroom).  Values
// outside the window (zeros aside), infinities and NaNs are added straight
// into the caller's copy with an FP32 atomic, as the reference adds every
// value.  lo is set per feature so that the window ends kWinMargin binades
// above the largest centroid coordinate of that feature: samples lie near
// their centroids, so nearly every value falls inside.
constexpr int kWinMargin = 4;
constexpr int kWinTopW = 20;   // weights: window up to 2^20

__device__ inline void window_add(unsigned long long *sum, float *fallback, int64_t off,
                                  float v, int lo, int W) {
  const unsigned b = __float_as_uint(v);
  const int sh = (int)((b >> 23) & 0xffu) - lo;
  if ((unsigned)sh <= (unsigned)W) {
    const unsigned long long m =
        (unsigned long long)((b & 0x7fffffu) | 0x800000u) << sh;
    atomicAdd(sum + off, (b >> 31) ? 0ull - m : m);
  } else if (v != 0.f) {
    atomicAdd(fallback + off, v);
  }
}

// Width W of the window when one block adds at most `count` values into one
// sum: 2^(24 + W) count < 2^63.
inline int window_width(int64_t count) {
  int bits = 0;
  while (bits < 40 && (int64_t(1) << bits) < count) ++bits;
  const int w = 38 - bits;
  return w < 1 ? 1 : w > 30 ? 30 : w;
}

// Lowest binade of the window whose largest value's binade is `e` (a
// centroid coordinate's, for a feature) and whose margin is `margin`.
__device__ inline int window_low(int e, int margin, int W) {
  const int top = e + margin;
  const int lo = top > W + 1 ? top : W + 1;
  return (lo < 254 ? lo : 254) - W;
}

}  // namespace kmd
