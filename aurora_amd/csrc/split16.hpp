// Pieces of the split-fp16 products (fp32 values as two fp16 numbers, summed by
// v_mfma_f32_16x16x32_f16) shared by the GEMM and the attention kernels.
#pragma once

#include "common.hpp"

namespace aursplit {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ floatx4 mfma_f16(half8 a, half8 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// 2^p as a float (−126 ≤ p ≤ 127).
__device__ __forceinline__ float exp_scale(int p) { return __uint_as_float((unsigned)(p + 127) << 23); }

// h = fp16(x·s), l = fp16(x·s − h) of two values.
__device__ __forceinline__ half2v split_high(float x0, float x1, float s0, float s1) {
  return __builtin_convertvector(float2v{x0 * s0, x1 * s1}, half2v);
}
__device__ __forceinline__ half2v split_low(float x0, float x1, float s0, float s1, half2v h) {
  return __builtin_convertvector(float2v{__builtin_fmaf(x0, s0, -(float)h[0]), __builtin_fmaf(x1, s1, -(float)h[1])}, half2v);
}
__device__ __forceinline__ void split2(float x0, float x1, float s0, float s1, half2v& h, half2v& l) {
  h = split_high(x0, x1, s0, s1);
  l = split_low(x0, x1, s0, s1, h);
}

constexpr float kSplitLimit = 65504.f;  // largest scaled magnitude let through
constexpr float kSplitFine = 0.0625f;   // smallest whose error, 2^-25, is below 2^-21 of it

// Is any |h| of N pairs outside [kSplitFine, kSplitLimit], zero, infinite or NaN?
// (2h − 2·0x2c00 in 16 bits, without the sign, is below 0xa000 for the others.)
typedef unsigned short ushort2v __attribute__((ext_vector_type(2)));
template <int N>
__device__ __forceinline__ ushort2v high_range(const half2v (&h)[N]) {
  ushort2v m = {0, 0};
#pragma unroll
  for (int e = 0; e < N; ++e) {
    ushort2v t;
    asm("v_pk_mad_u16 %0, %1, 2, %2 op_sel_hi:[1,0,1]" : "=v"(t) : "v"(h[e]), "s"(0xa800a800u));
    m = __builtin_elementwise_max(m, t);
  }
  return m;
}
__device__ __forceinline__ bool out_of_range(ushort2v t) { return max(t[0], t[1]) >= 0xa000; }

// Byte offset of granule q (8 k, 16 bytes) of row r in an LDS plane [ROWS][32]:
// q ^ t(r / 4), t = 0, 2, 3, 1.  A b128 access runs in four phases of 16 lanes
// (lanes 0-3, 12-15, 20-27 first; 4-11, 16-19, 28-31 next; then the same of
// the upper half), which for a fragment read are rows 0-3 and 12-15 of one
// octet with rows 4-11 of the next: with this t each phase covers the 64 banks
// once, as it does for the rows and octets of a store.
__device__ __forceinline__ int split_granule(int r, int q) {
  const int R = (r >> 2) & 3, t = (R >> 1) | (((R ^ (R >> 1)) & 1) << 1);
  return r * 64 + (q ^ t) * 16;
}

}  // namespace aursplit
