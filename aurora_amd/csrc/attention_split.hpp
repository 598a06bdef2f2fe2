// LDS layout and scales shared by the split-fp16 attention kernels.
#pragma once

#include "attention.hpp"
#include "split16.hpp"

namespace aurattn {

using namespace aursplit;

template <int DH>
struct SplitGeo {
  static constexpr int KS = (DH + 31) / 32;  // 32-wide steps over the head dimension
  static constexpr int DT = (DH + 15) / 16;  // 16-row tiles of Vᵀ / Oᵀ
  static constexpr int KROW = KS * 64;       // bytes of a K row in LDS
  static constexpr int KPLANE = 64 * KROW, VPLANE = DT * 16 * 128;
  // Small values among 16 rows of a tile that are one too many: a row of them has
  // DH, a column 16.  (N(0, 1) values have 0.01 on average, those with
  // columns 30 times the others' 0.3.)
  static constexpr int FINE = DH < 16 ? DH : 16;
};

// Granule q of row r in rows of 128 bytes: as split_granule, every phase of 16
// lanes covers the 64 banks once.
__device__ __forceinline__ int granule128(int r, int q) { return r * 128 + ((q ^ (r >> 1)) & 7) * 16; }
template <int ROW>
__device__ __forceinline__ int k_granule(int r, int q) {
  return ROW == 64 ? split_granule(r, q) : granule128(r, q);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int m = 8; m >= 1; m >>= 1) v = fmaxf(v, shfl_xor(v, m));
  return rows4_max(v);
}

// Lanes whose value x is not zero but too small for the scale s.
__device__ __forceinline__ int count_fine(float x, float s, bool in = true) {
  return __popcll(__ballot(in & (x != 0.f) & (fabsf(x) * s < kSplitFine)));
}

// p with max·2^p in [2^13, 2^14).
__device__ __forceinline__ int tile_exp(float m) { return min(140 - (int)(__float_as_uint(m) >> 23), 127); }

// p with max·2^p in [2^14, 2^15), for values whose small ones are counted.
__device__ __forceinline__ int value_exp(float m) { return min(141 - (int)(__float_as_uint(m) >> 23), 127); }

}  // namespace aurattn
