// Kernel arguments and the fused output forms shared by the GEMM kernels.
#pragma once

#include "common.hpp"

namespace aurgemm {

struct GemmArgs {
  const float* A;
  const float* B;
  float* C;
  float* P;  // split-K partials [splits][M][N]
  int M, N, K;
  int lda, ldb, ldc;
  int k_chunk;  // K range per blockIdx.z (multiple of BK)
  int split;    // 1: write partial tiles to P[z] (epilogue runs in splitk_reduce)
  int tiles_m, tiles_n;
  aur::Epilogue epi;
  // Strided batch (gridDim.y > 1): problem z uses A + z·sA, B + z·sB, C + z·sC.
  long long sA, sB, sC;
};

// Points the operands at problem blockIdx.y of a strided batch.
__device__ __forceinline__ void select_batch(GemmArgs& g) {
  if (gridDim.y > 1) {
    const long long z = blockIdx.y;
    g.A += z * g.sA;
    g.B += z * g.sB;
    g.C += z * g.sC;
  }
}

// Fused epilogue on one output element v = (A·B)(row, col), stored at C[i]
// with i = row*ldc + col (R, X, C2 share C's layout).
// GELU, tanh form (src/linalg.rs:72-87): gelu(x) = 0.5·x·(1 + tanh(u)),
// u = √(2/π)·(x + 0.044715·x³).  With σ(t) = 1/(1 + e^(−t)) the identities
// 1 + tanh(u) = 2σ(2u) and sech²(u) = 4σ(2u)(1 − σ(2u)) give both the value
// and the derivative from one exp2 and one reciprocal, with no cancellation:
//   gelu(x)  = x·σ(2u)
//   gelu'(x) = σ(2u) + 2x·σ(2u)(1 − σ(2u))·√(2/π)·(1 + 3·0.044715·x²)
// (1 − σ(2u) = e^(−2u)·σ(2u) where σ is near 1).  The tanhf form spends
// most of the FFN GEMM epilogues in VALU work.
__device__ __forceinline__ float gelu_sigma(float x, float& one_minus) {
  const float k = 0.7978845608028654f, log2e = 1.4426950408889634f;
  const float u = k * (x + 0.044715f * x * x * x);
  const float e = __builtin_amdgcn_exp2f(-2.0f * log2e * u);  // e^(−2u)
  const float sig = __builtin_amdgcn_rcpf(1.0f + e);
  one_minus = e < 1.0f ? e * sig : 1.0f - sig;
  return sig;
}

__device__ __forceinline__ float gelu_tanh(float x) {
  float om;
  return x * gelu_sigma(x, om);
}

__device__ __forceinline__ float gelu_tanh_grad(float x) {
  const float k = 0.7978845608028654f;
  float om;
  const float sig = gelu_sigma(x, om);
  return sig + 2.0f * x * sig * om * (k * (1.0f + 3.0f * 0.044715f * x * x));
}

__device__ __forceinline__ void apply_epilogue(const aur::Epilogue& e, float* __restrict__ C, size_t i,
                                               float v) {
  switch (e.mode) {
    case aur::EPI_ACCUM: C[i] = C[i] + v; break;
    case aur::EPI_RESID: C[i] = e.R[i] + v; break;
    case aur::EPI_GELU:
      C[i] = v;
      e.C2[i] = gelu_tanh(v);
      break;
    case aur::EPI_GELU_BWD: C[i] = v * gelu_tanh_grad(e.X[i]); break;
    default: C[i] = v; break;
  }
}

// Writes a wave's TM×TN grid of 16×16 accumulator tiles (lane holds rows
// 4·g16 + e, column l16 of each) with the epilogue mode fixed at compile
// time, so the store loops carry no per-element branch.  MODE −1: split-K
// partial tile into P[z].  `full`: every row and column is in range, and skip
// leaves out nothing.
struct SkipNone {
  __device__ __forceinline__ bool operator()(int, int, int) const { return false; }
};
template <int MODE, int TM, int TN, class Skip>
__device__ __forceinline__ void write_tile(const GemmArgs& g, const floatx4 (&acc)[TM][TN], int r0, int c0,
                                           int g16, int l16, bool full, Skip skip) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = c0 + j * 16 + l16;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = r0 + i * 16 + 4 * g16 + e;
        if (!full && (row >= g.M || col >= g.N || skip(i, j, e))) continue;
        const float v = acc[i][j][e];
        if constexpr (MODE < 0) {
          g.P[((size_t)blockIdx.z * g.M + row) * g.N + col] = v;
        } else {
          const size_t idx = (size_t)row * g.ldc + col;
          if constexpr (MODE == aur::EPI_ACCUM) g.C[idx] = g.C[idx] + v;
          else if constexpr (MODE == aur::EPI_RESID) g.C[idx] = g.epi.R[idx] + v;
          else if constexpr (MODE == aur::EPI_GELU) {
            g.C[idx] = v;
            g.epi.C2[idx] = gelu_tanh(v);
          } else if constexpr (MODE == aur::EPI_GELU_BWD) g.C[idx] = v * gelu_tanh_grad(g.epi.X[idx]);
          else g.C[idx] = v;
        }
      }
    }
}

template <int TM, int TN, class Skip = SkipNone>
__device__ __forceinline__ void write_tiles(const GemmArgs& g, const floatx4 (&acc)[TM][TN], int r0, int c0,
                                            int g16, int l16, bool full, Skip skip = Skip()) {
  if (g.split) {
    write_tile<-1>(g, acc, r0, c0, g16, l16, full, skip);
    return;
  }
  switch (g.epi.mode) {
    case aur::EPI_ACCUM: write_tile<aur::EPI_ACCUM>(g, acc, r0, c0, g16, l16, full, skip); break;
    case aur::EPI_RESID: write_tile<aur::EPI_RESID>(g, acc, r0, c0, g16, l16, full, skip); break;
    case aur::EPI_GELU: write_tile<aur::EPI_GELU>(g, acc, r0, c0, g16, l16, full, skip); break;
    case aur::EPI_GELU_BWD: write_tile<aur::EPI_GELU_BWD>(g, acc, r0, c0, g16, l16, full, skip); break;
    default: write_tile<aur::EPI_STORE>(g, acc, r0, c0, g16, l16, full, skip); break;
  }
}

// The epilogue operand (R or X, laid out like C) of a wave's TM×TN tiles,
// in the accumulator layout: pre[i][j][e] = S[r0 + 16i + 4·g16 + e][c0 + 16j + l16].
template <int TM, int TN>
__device__ __forceinline__ void load_epi_operand(const GemmArgs& g, floatx4 (&pre)[TM][TN], int r0, int c0,
                                                 int g16, int l16, int mode) {
  const float* src = mode == aur::EPI_RESID ? g.epi.R : g.epi.X;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        pre[i][j][e] = src[(size_t)(r0 + i * 16 + 4 * g16 + e) * g.ldc + c0 + j * 16 + l16];
}

// write_tile for whole tiles whose epilogue operand was prefetched.
template <int MODE, int TM, int TN>
__device__ __forceinline__ void write_tile_pre(const GemmArgs& g, const floatx4 (&acc)[TM][TN],
                                               const floatx4 (&pre)[TM][TN], int r0, int c0, int g16,
                                               int l16) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const size_t idx = (size_t)(r0 + i * 16 + 4 * g16 + e) * g.ldc + c0 + j * 16 + l16;
        if constexpr (MODE == aur::EPI_RESID)
          g.C[idx] = pre[i][j][e] + acc[i][j][e];
        else
          g.C[idx] = acc[i][j][e] * gelu_tanh_grad(pre[i][j][e]);
      }
}

}  // namespace aurgemm
