// Kernel arguments and row reductions shared by the attention kernels.
#pragma once

#include "common.hpp"

namespace aurattn {

constexpr int TQ = 64;  // rows per tile (4 waves × 16)
constexpr float LOG2E = 1.4426950408889634f;

struct AttnArgs {
  const float* q;
  const float* k;
  const float* v;
  const float* o;    // forward output (bwd pass 1)
  const float* dO;   // gradient of the output
  float* out;        // forward output
  float* lse;        // [B, H, T]
  float* D;          // [B, H, T] rowdot
  float* ds;         // [B, H, ntri] 64×64 dS tiles of the causal lower triangle (ds_slot)
  int ntri;          // nqt·(nqt+1)/2 tiles per (sequence, head)
  float* dq;
  float* dk;
  float* dv;
  int ld_qkv;        // row stride of q, k, v
  int ld_o;          // row stride of out / o / dO
  int ld_d;          // row stride of dq, dk, dv
  int T, H;
  float scale;       // 1/sqrt(d_head)
  int overwrite;     // backward: store dq/dk/dv instead of accumulating into them
};

__device__ __forceinline__ float shfl_xor(float v, int m) { return __shfl_xor(v, m, 64); }

// Max and sum over lanes l, l^16, l^32, l^48 (the four 16-lane rows), every
// lane getting the result.  v_permlane16_swap exchanges the odd rows of its
// first operand with the even rows of its second (v_permlane32_swap: the
// upper half with the lower half), so with both operands = v each lane ends
// up holding its own value and its partner row's: VALU only, no LDS round
// trip as with a bpermute.  Sums add (r0 + r1) + (r2 + r3) in every lane.
__device__ __forceinline__ float rows4_max(float v) {
  const unsigned u = __float_as_uint(v);
  auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
  const unsigned u2 = __float_as_uint(v);
  auto t = __builtin_amdgcn_permlane32_swap(u2, u2, false, false);
  return fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
}
__device__ __forceinline__ float rows4_sum(float v) {
  const unsigned u = __float_as_uint(v);
  auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = __uint_as_float(s[0]) + __uint_as_float(s[1]);
  const unsigned u2 = __float_as_uint(v);
  auto t = __builtin_amdgcn_permlane32_swap(u2, u2, false, false);
  return __uint_as_float(t[0]) + __uint_as_float(t[1]);
}

// Forward on the fp16 matrix cores (attention_split.hip), d_head a multiple of 8 up to 64.
void fwd_split(const AttnArgs& a, int b, int d_head, hipStream_t st);
// Backward pass 2 (dK, dV and the dS tiles) on them (attention_bwd_split.hip), d_head 24 to 64.
void bwd_dkv_split(const AttnArgs& a, int b, int d_head, hipStream_t st);

}  // namespace aurattn
