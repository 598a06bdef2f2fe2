// Causal attention backward, pass 2 (dK, dV and the dS tiles), with the products
// on the fp16 matrix cores: K, V, Q, dO, P and dS are split into two fp16
// numbers each (split16.hpp), three MFMAs per product.
//
// A block owns 128 keys of one (sequence, head), a wave 32 of them (two columns
// of 16), and walks the 64-query tiles from its diagonal on.  S = Q·Kᵀ and
// dP = dO·Vᵀ leave a lane with scores of one key, and its registers of 32
// queries are, as they lie, the B operand of dVᵀ += dOᵀ·P and dKᵀ += Qᵀ·dS: the
// queries 16·(i/4) + 4g + i%4 (i = 0..7) of lane group g.  Q and dO are split
// once and laid down twice in LDS, as [query][d] and, in that order, [d][query].
//
// Scales: K (times log2(e)/sqrt(d_head)) and V per key, Q and dO per tile, P and
// dS per key and 32 queries.  Queries of odd index and columns of odd index carry
// a minus sign in Q and dO, odd columns in K and V, odd queries in P and dS (the
// MFMA truncates downwards: so the error's sign alternates over the scores of a
// key and over its results).  Products are summed from zero per 32 queries and
// added to the fp32 sums by the VALU.
//
// A block whose results are not finite, or that met values too far apart for a
// tile's scale, computes its keys again with the fp32 MFMA before anything of dK and
// dV is written: scores beyond 2^12; among 16 queries of Q or dO, 16 or more values
// that are not zero but 2^18 or more below the tile's largest (a row or a column has
// as many); a largest value outside 2^±50.  Fewer small values than that keep an
// absolute error of 2^-40 of the tile's largest.  With all blocks computed again the
// backward of B16 H8 T1024 d_head 64 takes 590 µs, against 275 and the fp32 MFMA
// pass's 392.
//
// Per 16×16 scores the MFMAs take 384 cycles (2048 with the fp32 MFMA); the
// exponentials, the split of P and dS, this wave's share of Q's and dO's and the
// sums' update are about as many VALU cycles.  256 VGPRs and 64 KB of LDS leave
// two waves per SIMD, which hardly overlap the two.  Measured at B16 H8 T1024
// d_head 64, whole backward: 392 → 274 µs against the fp32 MFMA kernel; with the
// next tile's loads in registers under the products 301 (it spills); S and dP
// multiplied together before P is used 319.
#include "attention_dkv.hpp"
#include "attention_split.hpp"

#include <type_traits>

using namespace aurattn;

namespace {

constexpr int KB = 128;  // keys per block

// Largest value of a tile or row outside 2^±50, infinite or not.
__device__ __forceinline__ bool too_far(float m) { return m >= 0x1p50f || (m > 0.f && m < 0x1p-50f); }
// A scale's exponent for such a value in range (also the sum of two keeps 2^-p normal).
__device__ __forceinline__ int clamp_exp(int p) { return max(-37, min(63, p)); }

template <int DH>
struct DkvSplitLds {
  using G = SplitGeo<DH>;
  struct Split {
    char q[2 * G::KPLANE], o[2 * G::KPLANE];    // [query][d], h and l
    char qt[2 * G::VPLANE], ot[2 * G::VPLANE];  // [d][query], h and l
    float lse[TQ], D[TQ];
  };
  union {
    Split s;
    DkvLds<DH, 1> fp32;
  };
};

// Row krow of a head (columns 32c + 8g .. + 7 for c < KS) times `mul`, split at
// its own scale with odd columns negated.  Returns the scale's exponent.
template <int DH>
__device__ __forceinline__ int split_row(const float* row, float mul, int g, half8* hi, half8* lo, bool& far) {
  constexpr int KS = SplitGeo<DH>::KS;
  float x[KS][8], mx = 0.f;
#pragma unroll
  for (int c = 0; c < KS; ++c) {
    floatx4 u = {0.f, 0.f, 0.f, 0.f}, v = u;
    if (DH % 32 == 0 || 32 * c + 8 * g < DH) {
      u = *reinterpret_cast<const floatx4*>(row + 32 * c + 8 * g);
      v = *reinterpret_cast<const floatx4*>(row + 32 * c + 8 * g + 4);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) x[c][e] = u[e] * mul, x[c][4 + e] = v[e] * mul;
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[c][e]));
  }
  mx = rows4_max(mx);
  far |= too_far(mx);
  const int p = clamp_exp(tile_exp(mx));
  const float s = exp_scale(p);
#pragma unroll
  for (int c = 0; c < KS; ++c)
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      half2v hh, ll;
      split2(x[c][e], x[c][e + 1], s, -s, hh, ll);
      hi[c][e] = hh[0], hi[c][e + 1] = hh[1];
      lo[c][e] = ll[0], lo[c][e + 1] = ll[1];
    }
  return p;
}

template <int DH>
__global__ void __launch_bounds__(256, 2) mha_bwd_dkv_split_kernel(AttnArgs a) {
  using G = SplitGeo<DH>;
  constexpr int KS = G::KS, DT = G::DT;
  __shared__ __attribute__((aligned(1024))) DkvSplitLds<DH> lds;
  __shared__ float red[2][4];  // this tile's largest |Q| and |dO| of each wave
  __shared__ int again;        // the block's keys are to be computed in fp32
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int nqt = (a.T + TQ - 1) / TQ;
  const int kb = blockIdx.z;  // the first keys have the most work: dispatched first
  const int h = blockIdx.x, b = blockIdx.y;
  const int kw = kb * KB + 32 * w;  // this wave's first key
  const size_t row_base = (size_t)b * a.T;
  const float* Qb = a.q + row_base * a.ld_qkv + h * DH;
  const float* Kb = a.k + row_base * a.ld_qkv + h * DH;
  const float* Vb = a.v + row_base * a.ld_qkv + h * DH;
  const float* dOb = a.dO + row_base * a.ld_o + h * DH;
  const size_t stat = ((size_t)b * a.H + h) * a.T;
  float* ds_head = a.ds + ((size_t)b * a.H + h) * a.ntri * (TQ * TQ);

  // Staging: columns 2·vp, 2·vp + 1 of the queries of granule vg.
  const int vp = tid & 31, vg = tid >> 5;
  const int r0 = 32 * (vg >> 2) + 4 * (vg & 3);
  const bool live = 2 * vp < DH;
  float2v qx[8], ox[8];
  float r_lse = 0.f, r_D = 0.f;
  auto load = [&](int q0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      qx[i] = ox[i] = float2v{0.f, 0.f};
      const size_t row = min(q0 + r0 + 16 * (i >> 2) + (i & 3), a.T - 1);
      if (DH == 64 || live) {
        qx[i] = *reinterpret_cast<const float2v*>(Qb + row * a.ld_qkv + 2 * vp);
        ox[i] = *reinterpret_cast<const float2v*>(dOb + row * a.ld_o + 2 * vp);
      }
    }
    if (tid < TQ) {
      const int q = min(q0 + tid, a.T - 1);
      r_lse = a.lse[stat + q];
      r_D = a.D[stat + q];
    }
  };
  // The thread's values to both layouts of one tensor; true if too many of the wave's
  // 16 queries are too small for the tile's scale (SplitGeo::FINE).
  auto lay_down = [&](const float2v* x, int q0, int p, char* rows, char* cols) {
    const float s = exp_scale(p);
    half8 th[2], tl[2];
    half2v all[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      half2v hh, ll;
      split2(x[i][0], x[i][1], i & 1 ? -s : s, i & 1 ? s : -s, hh, ll);
      all[i] = hh;
      th[0][i] = hh[0], th[1][i] = hh[1];
      tl[0][i] = ll[0], tl[1][i] = ll[1];
      if (KS == 2 || 2 * vp < KS * 32) {
        char* r = rows + k_granule<G::KROW>(r0 + 16 * (i >> 2) + (i & 3), vp >> 2) + 4 * (vp & 3);
        *reinterpret_cast<half2v*>(r) = hh;
        *reinterpret_cast<half2v*>(r + G::KPLANE) = ll;
      }
    }
    if (DT == 4 || 2 * vp < DT * 16) {
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        char* c = cols + granule128(2 * vp + r, vg);
        *reinterpret_cast<half8*>(c) = th[r];
        *reinterpret_cast<half8*>(c + G::VPLANE) = tl[r];
      }
    }
    int n = 0;
    if (__any((DH == 64 || live) && out_of_range(high_range(all)))) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const bool in = q0 + r0 + 16 * (i >> 2) + (i & 3) < a.T;  // the others are copies of the last
        n += count_fine(x[i][0], s, in) + count_fine(x[i][1], s, in);
      }
    }
    return n >= G::FINE;
  };

  // K and V fragments: key column l16 of tile ki, octet g of step c.
  half8 kh[2][KS], kl[2][KS], vh[2][KS], vl[2][KS];
  int pk[2], pv[2];
  bool far = false;
#pragma unroll
  for (int ki = 0; ki < 2; ++ki) {
    const size_t row = min(kw + 16 * ki + l16, a.T - 1);
    pk[ki] = split_row<DH>(Kb + row * a.ld_qkv, a.scale * LOG2E, g, kh[ki], kl[ki], far);
    pv[ki] = split_row<DH>(Vb + row * a.ld_qkv, 1.f, g, vh[ki], vl[ki], far);
  }
  const int pk_min = min(pk[0], pk[1]);  // this lane's keys: see the score limit below
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  floatx4 acc_k[2][DT], acc_v[2][DT];
#pragma unroll
  for (int ki = 0; ki < 2; ++ki)
#pragma unroll
    for (int d = 0; d < DT; ++d) acc_k[ki][d] = acc_v[ki][d] = zero;
  if (tid == 0) again = 0;

  // 32 queries from 32·kk of the tile qt against the wave's keys.
  auto compute = [&](int qt, int kk, int pq, int po, auto diag) {
    constexpr bool DIAG = decltype(diag)::value;
    const int q0 = qt * TQ + 32 * kk;
    // 16 queries from 32·kk + 16·j of one tensor against the wave's keys
    auto product = [&](const char* rows, int j, const half8 (*bh)[KS], const half8 (*bl)[KS], floatx4* out) {
      out[0] = out[1] = zero;
#pragma unroll
      for (int c = 0; c < KS; ++c) {
        const char* at = rows + k_granule<G::KROW>(32 * kk + 16 * j + l16, 4 * c + g);
        const half8 h = *reinterpret_cast<const half8*>(at), l = *reinterpret_cast<const half8*>(at + G::KPLANE);
#pragma unroll
        for (int ki = 0; ki < 2; ++ki) out[ki] = mfma_f16(l, bh[ki][c], out[ki]);
#pragma unroll
        for (int ki = 0; ki < 2; ++ki) out[ki] = mfma_f16(h, bl[ki][c], out[ki]);
#pragma unroll
        for (int ki = 0; ki < 2; ++ki) out[ki] = mfma_f16(h, bh[ki][c], out[ki]);
      }
    };
    float p[2][8];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      floatx4 s_[2];
      product(lds.s.q, j, kh, kl, s_);
      const floatx4 lq = *reinterpret_cast<const floatx4*>(lds.s.lse + 32 * kk + 16 * j + 4 * g);
#pragma unroll
      for (int ki = 0; ki < 2; ++ki) {
        const float cs = exp_scale(-(pq + pk[ki]));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p[ki][4 * j + e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_[ki][e], e & 1 ? -cs : cs, -lq[e]));
          if (DIAG && kw + 16 * ki + l16 > q0 + 16 * j + 4 * g + e) p[ki][4 * j + e] = 0.f;
        }
      }
    }
    half8 xh[2], xl[2];
    float c[2];
    // y (values of this lane's two keys) as fp16 pairs, odd queries negated; px:
    // the scale of the tile it is multiplied with
    auto split_cols = [&](float (*y)[8], int px) {
#pragma unroll
      for (int ki = 0; ki < 2; ++ki) {
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(y[ki][i]));
        const int py = max(-60, min(126 - px, tile_exp(rows4_max(mx))));
        const float s = exp_scale(py);
        c[ki] = exp_scale(-(py + px));
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          half2v hh, ll;
          split2(y[ki][i], y[ki][i + 1], s, -s, hh, ll);
          xh[ki][i] = hh[0], xh[ki][i + 1] = hh[1];
          xl[ki][i] = ll[0], xl[ki][i + 1] = ll[1];
        }
      }
    };
    auto accumulate = [&](const char* cols, floatx4 (*acc)[DT]) {
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        const char* at = cols + granule128(16 * d + l16, 4 * kk + g);
        const half8 th = *reinterpret_cast<const half8*>(at), tl = *reinterpret_cast<const half8*>(at + G::VPLANE);
        floatx4 u[2] = {zero, zero};
#pragma unroll
        for (int ki = 0; ki < 2; ++ki) u[ki] = mfma_f16(tl, xh[ki], u[ki]);
#pragma unroll
        for (int ki = 0; ki < 2; ++ki) u[ki] = mfma_f16(th, xl[ki], u[ki]);
#pragma unroll
        for (int ki = 0; ki < 2; ++ki) u[ki] = mfma_f16(th, xh[ki], u[ki]);
#pragma unroll
        for (int ki = 0; ki < 2; ++ki)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[ki][d][e] = __builtin_fmaf(u[ki][e], c[ki], acc[ki][d][e]);
      }
    };
    split_cols(p, po);
    accumulate(lds.s.ot, acc_v);
    // P becomes dS, stored for the dQ pass in the layout of its tiles
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      floatx4 dp[2];
      product(lds.s.o, j, vh, vl, dp);
      const floatx4 Dq = *reinterpret_cast<const floatx4*>(lds.s.D + 32 * kk + 16 * j + 4 * g);
#pragma unroll
      for (int ki = 0; ki < 2; ++ki) {
        const float cp = exp_scale(-(po + pv[ki]));
        const int k16 = (kw >> 4) + ki, kt = k16 >> 2;
        float* tile = ds_head + (size_t)(qt * (qt + 1) / 2 + kt) * (TQ * TQ) + (k16 & 3) * (16 * TQ) + l16;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p[ki][4 * j + e] *= __builtin_fmaf(dp[ki][e], e & 1 ? -cp : cp, -Dq[e]);
          __builtin_nontemporal_store(p[ki][4 * j + e], &tile[(32 * kk + 16 * j + 2 * e + 8 * (g >> 1) + (g & 1)) * 16]);
        }
      }
    }
    split_cols(p, pq);
    accumulate(lds.s.qt, acc_k);
  };

  const int qt0 = kb * (KB / TQ);
  for (int qt = qt0; qt < nqt; ++qt) {
    const int q0 = qt * TQ;
    load(q0);
    float mq = 0.f, mo = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      mq = fmaxf(fmaxf(mq, fabsf(qx[i][0])), fabsf(qx[i][1]));
      mo = fmaxf(fmaxf(mo, fabsf(ox[i][0])), fabsf(ox[i][1]));
    }
    mq = wave_max(mq);
    mo = wave_max(mo);
    if (lane == 0) red[0][w] = mq, red[1][w] = mo;
    __syncthreads();  // the maxima are there, and every wave is done with the previous tile
    mq = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    mo = fmaxf(fmaxf(red[1][0], red[1][1]), fmaxf(red[1][2], red[1][3]));
    const int pq = clamp_exp(value_exp(mq)), po = clamp_exp(value_exp(mo));
    // Scores up to about 2^12 keep an absolute error of 2^-24 however small their
    // query is beside the tile's largest.
    far |= too_far(mq) || too_far(mo) || pq + pk_min < 17;
    far |= lay_down(qx, q0, pq, lds.s.q, lds.s.qt);
    far |= lay_down(ox, q0, po, lds.s.o, lds.s.ot);
    if (tid < TQ) {  // queries past T: P = exp2(S - inf) = 0
      lds.s.lse[tid] = q0 + tid < a.T ? r_lse * LOG2E : INFINITY;
      lds.s.D[tid] = q0 + tid < a.T ? r_D : 0.f;
    }
    __syncthreads();
#pragma unroll 1
    for (int kk = 0; kk < 2; ++kk) {
      const int qk = q0 + 32 * kk;
      if (qk + 31 < kw) {
        // All masked.  The diagonal tile's reader skips these 16-query blocks
        // too: it reads key blocks up to its own.
        continue;
      }
      if (qk >= kw + 31)
        compute(qt, kk, pq, po, std::false_type{});
      else
        compute(qt, kk, pq, po, std::true_type{});
    }
  }

#pragma unroll
  for (int ki = 0; ki < 2; ++ki)
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        far |= !(acc_k[ki][d][e] - acc_k[ki][d][e] == 0.f) || !(acc_v[ki][d][e] - acc_v[ki][d][e] == 0.f);
        if (e & 1) acc_k[ki][d][e] = -acc_k[ki][d][e], acc_v[ki][d][e] = -acc_v[ki][d][e];
      }
  if (far) again = 1;
  __syncthreads();  // also: every wave is done with the last tile
  if (again) {
#pragma unroll 1
    for (int kt = qt0; kt < min(qt0 + KB / TQ, nqt); ++kt) dkv_tile<DH, 1>(a, lds.fp32, kt, h, b);
    return;
  }
#pragma unroll
  for (int ki = 0; ki < 2; ++ki) {
    const int krow = kw + 16 * ki + l16;
    if (krow >= a.T) continue;
    float* dkr = a.dk + (row_base + krow) * a.ld_d + h * DH;
    float* dvr = a.dv + (row_base + krow) * a.ld_d + h * DH;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      if (DH % 16 != 0 && 16 * d + 4 * g >= DH) continue;
      floatx4* k4 = reinterpret_cast<floatx4*>(dkr + 16 * d + 4 * g);
      floatx4* v4 = reinterpret_cast<floatx4*>(dvr + 16 * d + 4 * g);
      *k4 = a.overwrite ? acc_k[ki][d] * a.scale : *k4 + acc_k[ki][d] * a.scale;
      *v4 = a.overwrite ? acc_v[ki][d] : *v4 + acc_v[ki][d];
    }
  }
}

template <int DH>
void launch(const AttnArgs& a, int b, hipStream_t st) {
  hipLaunchKernelGGL(mha_bwd_dkv_split_kernel<DH>, dim3(a.H, b, (a.T + KB - 1) / KB), dim3(256), 0, st, a);
}

}  // namespace

namespace aurattn {

void bwd_dkv_split(const AttnArgs& a, int b, int d_head, hipStream_t st) {
  switch (d_head) {
    case 24: launch<24>(a, b, st); break;
    case 32: launch<32>(a, b, st); break;
    case 40: launch<40>(a, b, st); break;
    case 48: launch<48>(a, b, st); break;
    case 56: launch<56>(a, b, st); break;
    default: launch<64>(a, b, st); break;
  }
}

}  // namespace aurattn
