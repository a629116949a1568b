// Entry points on sample-major rows (n, d), the layout an estimator's caller
// has: distances of rows to every centre without transposing X and the result.
#include <algorithm>

#include "common.hpp"

namespace kmd {

namespace {

constexpr int kRNT = 256;               // threads: 4 waves of 64 rows
constexpr int kRWaves = kRNT / kWave;
constexpr int kRC = 4;                  // centres whose chains run side by side

// padded[c][f] = centres[c][f], 0 outside: k rounded up to kRC rows of DB.
template <typename T>
__global__ void __launch_bounds__(kRNT)
    pad_centres_krn(int64_t k, int64_t d, int log2_db, int64_t total,
                    const T *__restrict__ C, T *__restrict__ padded) {
  const int64_t i = blockIdx.x * (int64_t)kRNT + threadIdx.x;
  if (i >= total) return;
  const int64_t c = i >> log2_db, f = i & ((1 << log2_db) - 1);
  padded[i] = (c < k && f < d) ? C[c * d + f] : T(0);
}

// D[s][c] = sqrt(sum_f (C[c][f] - X[s][f])^2), the chain over ascending f of
// fused multiply-adds as in the generic kernel's distances (lloyd.hip), so
// the same bits; padded features add (0 - 0)^2.
//
// One lane per row, its d values in registers; the centres are uniform in the
// wave and so come through the scalar cache as the subtraction's scalar
// operand.  Rows enter and results leave through a per-wave LDS tile (128
// bytes of 64 rows), so both sides of global memory move whole lines; no
// block barrier, the lanes of a wave exchange with wave_lds_order.
//
// Bound by the vector unit: two operations per (row, centre, feature) and no
// second unit to share them with (the expanded form on the matrix core would
// cancel).  n = 1,000,000, d = 32, k = 64: 0.104 ms of vector issue, 0.082 ms
// of memory; takes 0.180
// ms, a fifth of it in the correctly rounded square roots.  Two transposes around a feature-major kernel took
// 0.106 + 0.186 + 0.129 ms.
template <typename T, int DB>
__global__ void __launch_bounds__(kRNT)
    row_distances_krn(int64_t n, int d, int k, int span, const T *__restrict__ X,
                      const T *__restrict__ C, T *__restrict__ D) {
  constexpr int kRF = 128 / sizeof(T);   // features (and centres) per LDS tile
  __shared__ T tiles[kRWaves][kWave][kRF + 1];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  T(&tile)[kWave][kRF + 1] = tiles[wave];
  const int64_t s0 = ((int64_t)blockIdx.x * kRWaves + wave) * kWave;
  if (s0 >= n) return;
  const int rows = (int)min<int64_t>(kWave, n - s0);
  // 256 or 512 bytes of whole rows' pieces per wave access
  const int tx = lane & (kRF - 1), ty = lane / kRF;
  constexpr int kTY = kWave / kRF;

  T x[DB];
#pragma unroll
  for (int f0 = 0; f0 < DB; f0 += kRF) {
    constexpr int kW = DB < kRF ? DB : kRF;   // values of this pass
#pragma unroll 8
    for (int r = ty; r < kWave; r += kTY)
      tile[r][tx] = (r < rows && f0 + tx < d) ? X[(s0 + r) * d + f0 + tx] : T(0);
    wave_lds_order();
#pragma unroll
    for (int f = 0; f < kW; ++f) x[f0 + f] = tile[lane][f];
    wave_lds_order();
  }
  // this block's centres (span: a multiple of kRF)
  const int c1 = (int)min<int64_t>(k, (int64_t)(blockIdx.y + 1) * span);
  for (int c0 = blockIdx.y * span; c0 < c1; c0 += kRF) {
    const int m = min(kRF, c1 - c0);
    for (int c = 0; c < m; c += kRC) {
      const T *row = C + (int64_t)(c0 + c) * DB;
      T acc[kRC];
#pragma unroll
      for (int j = 0; j < kRC; ++j) acc[j] = T(0);
#pragma unroll
      for (int f = 0; f < DB; ++f) {
#pragma unroll
        for (int j = 0; j < kRC; ++j) {
          const T diff = row[j * DB + f] - x[f];
          acc[j] = fma(diff, diff, acc[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < kRC; ++j) tile[lane][c + j] = sqrt(acc[j]);
    }
    wave_lds_order();
#pragma unroll 8
    for (int r = ty; r < kWave; r += kTY)
      if (r < rows && tx < m) D[(s0 + r) * k + c0 + tx] = tile[r][tx];
    wave_lds_order();
  }
}

// Register rows: d rounded up to 8, 16, 32, 64 or (float) 128; 0: not served.
template <typename T>
int row_bucket(int64_t d) {
  for (int b : {8, 16, 32, 64, 128})
    if (d <= b) return (sizeof(T) == 8 && b == 128) ? 0 : b;
  return 0;
}

}  // namespace

template <typename T>
int64_t row_distances_scratch(int64_t d, int64_t k) {
  return ceil_div<int64_t>(k, kRC) * kRC * row_bucket<T>(d);
}

template <typename T>
void launch_row_distances(int64_t n, int64_t d, int64_t k, const T *X, const T *C,
                          T *scratch, T *D, hipStream_t s) {
  if (n <= 0) return;
  const int DB = row_bucket<T>(d);
  require(DB > 0, "row distances: too many features");
  const int64_t total = row_distances_scratch<T>(d, k);
  const int64_t blocks = ceil_div<int64_t>(n, kRNT);
  require(blocks <= INT32_MAX && ceil_div<int64_t>(total, kRNT) <= INT32_MAX,
          "row distances: array too large");
  hipLaunchKernelGGL(pad_centres_krn<T>, dim3((unsigned)ceil_div<int64_t>(total, kRNT)),
                     dim3(kRNT), 0, s, k, d, __builtin_ctz(DB), total, C, scratch);
  KMD_LAUNCH_CHECK();
  // Few rows leave most of the chip idle while a lane goes through all centres: then
  // the centres are split over blocks too, up to two blocks per CU in all (float64,
  // d = 17, k = 200: n = 2000 193 -> 81 us, n = 30,000 200 -> 116; the two transposes
  // and the feature-major kernel 168 and 180).
  constexpr int64_t kRF = 128 / sizeof(T);
  const int64_t tiles = ceil_div<int64_t>(k, kRF);
  const int64_t want = std::max<int64_t>(
      1, std::min<int64_t>(std::min<int64_t>(tiles, 65535), 2 * device_cu_count() / blocks));
  const int64_t span = ceil_div<int64_t>(tiles, want) * kRF;
  const dim3 grid((unsigned)blocks, (unsigned)ceil_div<int64_t>(k, span));
  auto run = [&](auto bucket) {
    if constexpr (sizeof(T) == 4 || bucket() <= 64)
      hipLaunchKernelGGL((row_distances_krn<T, bucket()>), grid, dim3(kRNT), 0, s, n, (int)d,
                         (int)k, (int)span, X, (const T *)scratch, D);
  };
  switch (DB) {
    case 8: run(std::integral_constant<int, 8>{}); break;
    case 16: run(std::integral_constant<int, 16>{}); break;
    case 32: run(std::integral_constant<int, 32>{}); break;
    case 64: run(std::integral_constant<int, 64>{}); break;
    default: run(std::integral_constant<int, 128>{});
  }
  KMD_LAUNCH_CHECK();
}

#define KMD_INST_ROWS(T)                                                       \
  template int64_t row_distances_scratch<T>(int64_t, int64_t);                 \
  template void launch_row_distances<T>(int64_t, int64_t, int64_t, const T *,  \
                                        const T *, T *, T *, hipStream_t);
KMD_INST_ROWS(float)
KMD_INST_ROWS(double)

}  // namespace kmd
