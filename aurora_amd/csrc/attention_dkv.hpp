// Tiles of the attention kernels in fp32 and the fp32 dK/dV pass over one key
// tile, which the split-fp16 pass takes too where its scales would not hold.
#pragma once

#include "attention.hpp"

namespace aurattn {

template <int DH>
struct Geo {
  static constexpr int NC = (DH + 15) / 16;  // 16-wide chunks of the head dim
  static constexpr int LDT = NC * 16 + 4;    // padded LDS row stride (floats)
  static constexpr int TILE = TQ * LDT;
  static constexpr int F4 = TQ * DH / 4;     // float4 per [64 × DH] tile
  static constexpr int NV = (F4 + 255) / 256;
  // Does a float4 at head-dim offset `d` hold real data?
  __device__ static __forceinline__ bool live(int d) { return DH % 16 == 0 || d < DH; }
};

// A [64 rows × DH] fp32 tile (rows r0.., zero-filled at r >= T) copied from a
// row-major source with row stride ld into registers, then into LDS.  LDS
// columns past DH (DH = 8) are zero-filled once by zero_pad_cols.
template <int DH>
struct TileRegs {
  using G = Geo<DH>;
  floatx4 v[G::NV];
  int r0 = 0, T = 0;  // of the last load: rows r0 + r ≥ T are stored as zeros
  // Branch-free, and nothing consumes the loaded values before store(): a
  // row past T is read from row T − 1 (in range) and zeroed only when stored,
  // so the loads stay in flight under whatever runs in between.
  __device__ __forceinline__ void load(const float* __restrict__ base, int ld, int r0_, int T_,
                                       int tid) {
    r0 = r0_;
    T = T_;
#pragma unroll
    for (int i = 0; i < G::NV; ++i) {
      const int f = tid + i * 256;
      const int r = f / (DH / 4), c = (f % (DH / 4)) * 4;
      if (G::F4 % 256 == 0 || f < G::F4)
        v[i] = *reinterpret_cast<const floatx4*>(base + (size_t)min(r0 + r, T - 1) * ld + c);
    }
  }
  __device__ __forceinline__ void store(float* __restrict__ s, int tid) const {
#pragma unroll
    for (int i = 0; i < G::NV; ++i) {
      const int f = tid + i * 256;
      const int r = f / (DH / 4), c = (f % (DH / 4)) * 4;
      if (G::F4 % 256 == 0 || f < G::F4) {
        const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<floatx4*>(s + r * G::LDT + c) = r0 + r < T ? v[i] : zero;
      }
    }
  }
};

template <int DH>
__device__ __forceinline__ void zero_pad_cols(float* s, int tid) {
  using G = Geo<DH>;
  if (DH % 16 != 0) {
    for (int i = tid; i < TQ * (G::NC * 16 - DH); i += 256) {
      const int r = i / (G::NC * 16 - DH), c = DH + i % (G::NC * 16 - DH);
      s[r * G::LDT + c] = 0.f;
    }
  }
}

// This lane's operand values of a 16-row slab:
// f[c][s] = X[row][16c + 4·(lane/16) + s]  (zero past DH or at row >= T).
template <int DH>
__device__ __forceinline__ void load_rows_frag(floatx4* f, const float* __restrict__ base, int ld,
                                               int row, int T, int g) {
#pragma unroll
  for (int c = 0; c < Geo<DH>::NC; ++c) {
    floatx4 x = {0.f, 0.f, 0.f, 0.f};
    if (row < T && Geo<DH>::live(16 * c + 4 * g))
      x = *reinterpret_cast<const floatx4*>(base + (size_t)row * ld + 16 * c + 4 * g);
    f[c] = x;
  }
}

// ---------------------------------------- backward pass 2: dK, dV (and dS)
// NS: LDS stages for the Q / dO tiles (staged through registers).  NS = 1 is
// compiled for three waves per SIMD and is the default (measured on MI355X at
// C2: backward 0.431 ms against 0.449 ms for the two-stage ring, which leaves
// two waves per SIMD).
template <int DH, int NS>
struct DkvLds {
  float tile[NS][2][Geo<DH>::TILE];  // [stage][Q,dO]
  float lse[NS][TQ];
  float D[NS][TQ];
};
// Key tile kt of head h of sequence b, by a block of 256 threads.  Ends with a barrier.
template <int DH, int NS>
__device__ __forceinline__ void dkv_tile(const AttnArgs& a, DkvLds<DH, NS>& lds, int kt, int h, int b) {
  using G = Geo<DH>;
  constexpr int NC = G::NC, LDT = G::LDT;
  auto& sm = lds.tile;
  auto& st_lse = lds.lse;
  auto& st_D = lds.D;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int nqt = (a.T + TQ - 1) / TQ;
  const int k0 = kt * TQ;
  const size_t row_base = (size_t)b * a.T;
  const float* Qb = a.q + row_base * a.ld_qkv + h * DH;
  const float* Kb = a.k + row_base * a.ld_qkv + h * DH;
  const float* Vb = a.v + row_base * a.ld_qkv + h * DH;
  const float* dOb = a.dO + row_base * a.ld_o + h * DH;
  const size_t stat = ((size_t)b * a.H + h) * a.T;

  const int krow = k0 + 16 * w + l16;  // this lane's key (column of S)
  floatx4 kf[NC], vf[NC];
  load_rows_frag<DH>(kf, Kb, a.ld_qkv, krow, a.T, g);
  load_rows_frag<DH>(vf, Vb, a.ld_qkv, krow, a.T, g);
  // K pre-multiplied by scale·log2(e): S comes out in the log2 domain.  dK
  // is accumulated from the unscaled dS and scaled once at the end.
  const float sl2 = a.scale * LOG2E;
#pragma unroll
  for (int c = 0; c < NC; ++c) kf[c] *= sl2;

  floatx4 acc_k[NC], acc_v[NC];
#pragma unroll
  for (int d = 0; d < NC; ++d) {
    acc_k[d] = floatx4{0.f, 0.f, 0.f, 0.f};
    acc_v[d] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  for (int st = 0; st < NS; ++st) {
    zero_pad_cols<DH>(sm[st][0], tid);
    zero_pad_cols<DH>(sm[st][1], tid);
  }
  TileRegs<DH> rq, rd;
  // The next tile's row statistics, raw: scaled and masked only when stored,
  // so no wait for them (and, the load counter being in order, for the
  // tile loads before them) at the top of the tile.
  float r_lse = 0.f, r_D = 0.f;
  int r_q = 0;
  auto load_stats = [&](int q0) {
    if (tid < TQ) {
      r_q = q0 + tid;
      const int qc = min(r_q, a.T - 1);
      r_lse = a.lse[stat + qc];
      r_D = a.D[stat + qc];
    }
  };
  rq.load(Qb, a.ld_qkv, k0, a.T, tid);
  rd.load(dOb, a.ld_o, k0, a.T, tid);
  load_stats(k0);
  rq.store(sm[0][0], tid);
  rd.store(sm[0][1], tid);
  if (tid < TQ) {
    st_lse[0][tid] = r_q < a.T ? r_lse * LOG2E : 0.f;
    st_D[0][tid] = r_q < a.T ? r_D : 0.f;
  }
  __syncthreads();

  for (int qt = kt; qt < nqt; ++qt) {
    const int cur = NS == 2 ? ((qt - kt) & 1) : 0;
    const bool more = qt + 1 < nqt;
    if (more) {
      rq.load(Qb, a.ld_qkv, (qt + 1) * TQ, a.T, tid);
      rd.load(dOb, a.ld_o, (qt + 1) * TQ, a.T, tid);
      load_stats((qt + 1) * TQ);
    }
    const float* Qs = sm[cur][0];
    const float* dOs = sm[cur][1];
    const int q0 = qt * TQ;
    float* ds_tile = a.ds + (((size_t)b * a.H + h) * a.ntri + qt * (qt + 1) / 2 + kt) * (TQ * TQ);
    // Query sub-tiles jq < w of the diagonal tile lie entirely before this
    // wave's keys: fully masked.
    const int jmin = (qt == kt) ? w : 0;
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      if (jq < jmin) continue;
      floatx4 s_ = {0.f, 0.f, 0.f, 0.f}, dp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const floatx4 qv = *reinterpret_cast<const floatx4*>(Qs + (16 * jq + l16) * LDT + 16 * c + 4 * g);
        const floatx4 dv_ = *reinterpret_cast<const floatx4*>(dOs + (16 * jq + l16) * LDT + 16 * c + 4 * g);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          s_ = mfma16x16x4(qv[s], kf[c][s], s_);   // S[q][key]
          dp = mfma16x16x4(dv_[s], vf[c][s], dp);  // dP[q][key]
        }
      }
      const floatx4 lq = *reinterpret_cast<const floatx4*>(&st_lse[cur][16 * jq + 4 * g]);
      const floatx4 Dq = *reinterpret_cast<const floatx4*>(&st_D[cur][16 * jq + 4 * g]);
      floatx4 p, ds;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int q = q0 + 16 * jq + 4 * g + e;
        float pe = __builtin_amdgcn_exp2f(s_[e] - lq[e]);
        if (qt == kt && krow > q) pe = 0.f;
        p[e] = pe;
        ds[e] = pe * (dp[e] - Dq[e]);
        // dS tile (qt, kt) for the dQ pass, in the ds_slot layout (this
        // wave's key block; row 4g + e in slot ds_slot(4g + e)).  Streamed
        // (non-temporal): it is read back only after the whole pass, and
        // keeping it out of L2 leaves room for the Q / dO tiles this block
        // and its neighbours re-read.
        __builtin_nontemporal_store(
            ds[e], &ds_tile[w * (16 * TQ) + (16 * jq + 2 * e + 8 * (g >> 1) + (g & 1)) * 16 + l16]);
      }
      // dVᵀ[d][key] += dOᵀ[d][q]·P[q][key];  dKᵀ[d][key] += Qᵀ[d][q]·dS[q][key]
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const float* dor = dOs + (16 * jq + 4 * g + s) * LDT + l16;
        const float* qr = Qs + (16 * jq + 4 * g + s) * LDT + l16;
#pragma unroll
        for (int d = 0; d < NC; ++d) {
          acc_v[d] = mfma16x16x4(dor[16 * d], p[s], acc_v[d]);
          acc_k[d] = mfma16x16x4(qr[16 * d], ds[s], acc_k[d]);
        }
      }
    }
    if (more) {
      if (NS == 1) __syncthreads();  // every wave is done with the only stage
      rq.store(sm[(cur + 1) % NS][0], tid);
      rd.store(sm[(cur + 1) % NS][1], tid);
      if (tid < TQ) {
        st_lse[(cur + 1) % NS][tid] = r_q < a.T ? r_lse * LOG2E : 0.f;
        st_D[(cur + 1) % NS][tid] = r_q < a.T ? r_D : 0.f;
      }
    }
    __syncthreads();
  }
  if (krow < a.T) {
    float* dkr = a.dk + (row_base + krow) * a.ld_d + h * DH;
    float* dvr = a.dv + (row_base + krow) * a.ld_d + h * DH;
#pragma unroll
    for (int d = 0; d < NC; ++d) {
      if (!G::live(16 * d + 4 * g)) continue;
      floatx4* pk = reinterpret_cast<floatx4*>(dkr + 16 * d + 4 * g);
      floatx4* pv = reinterpret_cast<floatx4*>(dvr + 16 * d + 4 * g);
      *pk = a.overwrite ? acc_k[d] * a.scale : *pk + acc_k[d] * a.scale;
      *pv = a.overwrite ? acc_v[d] : *pv + acc_v[d];
    }
  }
}

}  // namespace aurattn
