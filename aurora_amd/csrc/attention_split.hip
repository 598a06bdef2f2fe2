// Causal attention forward with the products on the fp16 matrix cores: Q, K, V
// and P are split into two fp16 numbers each (split16.hpp, gemm_split.hip), three
// MFMAs per product.
//
// A block owns 128 queries of one (sequence, head), a wave 32 of them (two
// columns of 16), and walks the 64-key tiles up to the diagonal.  Scores are
// computed transposed (Sᵀ = K·Qᵀ), so a lane holds scores of one query and its
// Sᵀ registers of 32 keys are, as they lie, the B operand of Oᵀ += Vᵀ·Pᵀ: the
// keys 16·(i/4) + 4g + i%4 (i = 0..7) of lane group g, in which order V is laid
// down in LDS.  K lies there as [key][d], V as [d][key], h and l planes each.
//
// Scales: Q (times log2(e)/sqrt(d_head)) per query, K per tile, V by a scale
// that only falls from tile to tile (the running sum is rescaled with the
// softmax correction), P by 2^14 times a power of two per query and tile that
// brings its largest value there to ½ … 1 (the small P of a later tile may meet
// larger V: with 2^14 alone the error was 2.8e-5 for V growing by 2^24); the
// scores' factors go into the exp2 argument's FMA.
// Odd keys of K and odd columns of V are scaled by the negative (the MFMA
// truncates downwards: so the error's sign alternates over a row's scores, and
// over its results).
// The largest value of a tile is found while it lies in registers, one LDS word
// per wave crossing the barrier that the tile's stage needs anyway.  A tile's
// V·P products are summed from zero and added to the corrected sum by the VALU.
// Queries whose result is not finite, and blocks that met an infinity in a tile
// or values too far apart for the scales, are computed again with the fp32 MFMA:
// scores beyond 2^12; among 16 keys of V, 16 or more values (d_head if that is less:
// as many as a row or a column has) that are not zero but 2^18 or more below the
// tile's largest; a V that grows by more than 2^60 from the first tile on.  Fewer
// small values than that keep an absolute error of 2^-40 of the tile's largest.
// With all blocks computed again B16 H8 T1024 d_head 64 takes 380 µs, against 85
// and the fp32 MFMA kernel's 150.
//
// Per 16×16 scores the MFMAs take 192 cycles (1024 with the fp32 MFMA), the
// softmax, the split of P and this wave's share of K's and V's about 300 VALU
// cycles; the sum of the two bounds it (the waves of a SIMD hardly overlap
// them).  Measured at B16 H8 T1024 d_head 64: 152 → 78 µs against the fp32 MFMA
// kernel; 16 queries per wave in 8-wave blocks (twice the LDS reads): 93; two
// LDS stages with one barrier per tile: 78.
#include "attention.hpp"
#include "attention_split.hpp"
#include "common.hpp"
#include "split16.hpp"

#include <type_traits>

using namespace aurattn;
using namespace aursplit;

namespace {

constexpr int QB = 128;             // queries per block
constexpr float kPScale = 16384.f;  // P ≤ 1 is split at this scale and 2^r, r ≤ kPExpMax
constexpr int kPExpMax = 60;

// The exponent for Q and K: at most 63, so that 2^-(pq + pk) is a normal number also
// where both are zero (a masked score is an infinity times it).
__device__ __forceinline__ int score_exp(float m) { return min(tile_exp(m), 63); }

// The 16 queries from q16 of one head again, with the fp32 MFMA and operands
// straight from memory (see the head of the file).
template <int DH>
__device__ void fwd_fp32_rows(const AttnArgs& a, const float* Qb, const float* Kb, const float* Vb, size_t row_base,
                              int b, int h, int q16, int g, int l16) {
  constexpr int NC = SplitGeo<DH>::DT;
  const int qrow = q16 + l16;
  const float sl2 = a.scale * LOG2E;
  auto live = [](int d) { return DH % 16 == 0 || d < DH; };
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  auto row4 = [&](const float* X, int row, int d) {
    return live(d) ? *reinterpret_cast<const floatx4*>(X + (size_t)min(row, a.T - 1) * a.ld_qkv + d) : zero;
  };
  floatx4 acc[NC];
#pragma unroll
  for (int d = 0; d < NC; ++d) acc[d] = zero;
  float m = -INFINITY, l = 0.f;
#pragma unroll 1
  for (int k16 = 0; k16 <= q16; k16 += 16) {
    floatx4 st = zero;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const floatx4 kf = row4(Kb, k16 + l16, 16 * c + 4 * g), qf = row4(Qb, qrow, 16 * c + 4 * g) * sl2;
#pragma unroll
      for (int s = 0; s < 4; ++s) st = mfma16x16x4(kf[s], qf[s], st);
    }
    if (k16 == q16) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * g + e > l16) st[e] = -INFINITY;
    }
    const float m_new = fmaxf(m, rows4_max(fmaxf(fmaxf(st[0], st[1]), fmaxf(st[2], st[3]))));
    const float alpha = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
    float ps = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      st[e] = __builtin_amdgcn_exp2f(st[e] - m_new);
      ps += st[e];
    }
    l = l * alpha + ps;
#pragma unroll
    for (int d = 0; d < NC; ++d) {
      acc[d] *= alpha;
      const int col = 16 * d + l16;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const float v = live(col) ? Vb[(size_t)min(k16 + 4 * g + s, a.T - 1) * a.ld_qkv + col] : 0.f;
        acc[d] = mfma16x16x4(v, st[s], acc[d]);
      }
    }
  }
  l = rows4_sum(l);
  if (qrow < a.T) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    float* orow = a.out + (row_base + qrow) * a.ld_o + h * DH;
#pragma unroll
    for (int d = 0; d < NC; ++d)
      if (live(16 * d + 4 * g)) *reinterpret_cast<floatx4*>(orow + 16 * d + 4 * g) = acc[d] * inv;
    if (g == 0) a.lse[((size_t)b * a.H + h) * a.T + qrow] = (m + __log2f(l)) * (1.f / LOG2E);
  }
}

template <int DH>
__global__ void __launch_bounds__(256, 2) mha_fwd_split_kernel(AttnArgs a) {
  using G = SplitGeo<DH>;
  constexpr int KS = G::KS, DT = G::DT;
  __shared__ __attribute__((aligned(1024))) char ks[2 * G::KPLANE];
  __shared__ __attribute__((aligned(1024))) char vs[2 * G::VPLANE];
  __shared__ float red[2][4];  // this tile's largest |K| and |V| of each wave
  __shared__ int wide;         // too many values of V far below their tile's largest were met
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int nqb = (a.T + QB - 1) / QB;
  const int qb = nqb - 1 - blockIdx.z;  // longest query blocks first over the whole launch
  const int h = blockIdx.x, b = blockIdx.y;
  const int q0 = qb * QB + 32 * w;  // this wave's first query
  const size_t row_base = (size_t)b * a.T;
  const float* Qb = a.q + row_base * a.ld_qkv + h * DH;
  const float* Kb = a.k + row_base * a.ld_qkv + h * DH;
  const float* Vb = a.v + row_base * a.ld_qkv + h * DH;

  // K: row kr, octets (tid & 3) + 4i.  V: columns 2·vp, 2·vp + 1 of granule vg
  // (keys 32·(vg/4) + 16·(i/4) + 4·(vg%4) + i%4).
  const int kr = tid >> 2, vp = tid & 31, vg = tid >> 5;
  const bool v_on = 2 * vp < DT * 16, v_live = 2 * vp < DH;
  float kx[KS][8], vx[2][8];
  auto load = [&](int k0) {
    const float* krow = Kb + (size_t)min(k0 + kr, a.T - 1) * a.ld_qkv;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int c = 8 * ((tid & 3) + 4 * i);
      floatx4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
      if (DH % 32 == 0 || c < DH) {
        x = *reinterpret_cast<const floatx4*>(krow + c);
        y = *reinterpret_cast<const floatx4*>(krow + c + 4);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) kx[i][e] = x[e], kx[i][4 + e] = y[e];
    }
    const int key = k0 + 32 * (vg >> 2) + 4 * (vg & 3);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float2v x = {0.f, 0.f};
      if (DH == 64 || v_live)
        x = *reinterpret_cast<const float2v*>(Vb + (size_t)min(key + 16 * (i >> 2) + (i & 3), a.T - 1) * a.ld_qkv + 2 * vp);
      vx[0][i] = x[0], vx[1][i] = x[1];
    }
  };

  // Q fragments: query column l16 of tile qi, octet g of step c.
  half8 qh[2][KS], ql[2][KS];
  int pq[2];
  const float sl2 = a.scale * LOG2E;
#pragma unroll
  for (int qi = 0; qi < 2; ++qi) {
    float x[KS][8], mx = 0.f;
    const float* qrow = Qb + (size_t)min(q0 + 16 * qi + l16, a.T - 1) * a.ld_qkv;
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      floatx4 u = {0.f, 0.f, 0.f, 0.f}, v = u;
      if (DH % 32 == 0 || 32 * c + 8 * g < DH) {
        u = *reinterpret_cast<const floatx4*>(qrow + 32 * c + 8 * g);
        v = *reinterpret_cast<const floatx4*>(qrow + 32 * c + 8 * g + 4);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) x[c][e] = u[e] * sl2, x[c][4 + e] = v[e] * sl2;
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[c][e]));
    }
    pq[qi] = score_exp(rows4_max(mx));
    const float s = exp_scale(pq[qi]);
#pragma unroll
    for (int c = 0; c < KS; ++c)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        half2v hh, ll;
        split2(x[c][e], x[c][e + 1], s, s, hh, ll);
        qh[qi][c][e] = hh[0], qh[qi][c][e + 1] = hh[1];
        ql[qi][c][e] = ll[0], ql[qi][c][e + 1] = ll[1];
      }
  }

  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  floatx4 acc[2][DT];
  float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
  int pr[2] = {0, 0};  // the exponent r of P in the last tile: of the sums too
#pragma unroll
  for (int qi = 0; qi < 2; ++qi)
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[qi][d] = zero;
  int pv = 127, pva = 127;  // V's scale so far, and when this wave last added to its sums
  int pv_top = -127;        // V's scale in the first tile that is not zero
  bool again = false;  // the block met an infinity, or values too far apart for a tile's scale
  // Scores up to about 2^12 keep an absolute error of 2^-24 however small their
  // key is beside the tile's largest; beyond that the fp32 MFMA computes them.
  int pq_min = min(pq[0], pq[1]);
#pragma unroll
  for (int i = 8; i >= 1; i >>= 1) pq_min = min(pq_min, __shfl_xor(pq_min, i, 64));
  if (tid == 0) wide = 0;

  // Scores, softmax and V·P of the wave's two query columns against the tile at
  // k0.  DIAG: sub-tiles of 16 keys past a query tile are skipped, the one on it
  // masked.
  auto compute = [&](int k0, int pk, float vcorr, auto diag) {
    constexpr bool DIAG = decltype(diag)::value;
    const int jd = DIAG ? (q0 - k0) / 16 : 4;  // sub-tile on column 0's diagonal; column 1's is the next
    floatx4 st[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      st[0][j] = st[1][j] = zero;
      if (DIAG && j > jd + 1) continue;
      half8 kh[KS], kl[KS];
#pragma unroll
      for (int c = 0; c < KS; ++c) {
        const char* p = ks + k_granule<G::KROW>(16 * j + l16, 4 * c + g);
        kh[c] = *reinterpret_cast<const half8*>(p);
        kl[c] = *reinterpret_cast<const half8*>(p + G::KPLANE);
      }
#pragma unroll
      for (int c = 0; c < KS; ++c)
#pragma unroll
        for (int qi = 0; qi < 2; ++qi) st[qi][j] = mfma_f16(kl[c], qh[qi][c], st[qi][j]);
#pragma unroll
      for (int c = 0; c < KS; ++c)
#pragma unroll
        for (int qi = 0; qi < 2; ++qi) st[qi][j] = mfma_f16(kh[c], ql[qi][c], st[qi][j]);
#pragma unroll
      for (int c = 0; c < KS; ++c)
#pragma unroll
        for (int qi = 0; qi < 2; ++qi) st[qi][j] = mfma_f16(kh[c], qh[qi][c], st[qi][j]);
    }
    half8 ph[2][2], pl[2][2];
    float av[2];
#pragma unroll
    for (int qi = 0; qi < 2; ++qi) {
      if (DIAG) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (j > jd + qi || (j == jd + qi && 4 * g + e > l16)) st[qi][j][e] = e & 1 ? INFINITY : -INFINITY;
      }
      // odd keys carry a minus sign
      float mx = fmaxf(fmaxf(st[qi][0][0], -st[qi][0][1]), fmaxf(st[qi][0][2], -st[qi][0][3]));
#pragma unroll
      for (int j = 1; j < 4; ++j)
        mx = fmaxf(mx, fmaxf(fmaxf(st[qi][j][0], -st[qi][j][1]), fmaxf(st[qi][j][2], -st[qi][j][3])));
      const float c = ldexpf(1.f, -(pq[qi] + pk));
      const float m_tile = rows4_max(mx) * c, m_new = fmaxf(m[qi], m_tile);
      const float alpha = __builtin_amdgcn_exp2f(m[qi] - m_new);
      m[qi] = m_new;
      const int r = (int)fminf(m_new - m_tile, (float)kPExpMax);
      const float at = (float)r - m_new;
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[qi][j][e], c, at));
          const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[qi][j][e + 1], -c, at));
          ps += p0 + p1;
          half2v hh, ll;
          split2(p0, p1, kPScale, kPScale, hh, ll);
          const int i = 4 * (j & 1) + e;
          ph[qi][j >> 1][i] = hh[0], ph[qi][j >> 1][i + 1] = hh[1];
          pl[qi][j >> 1][i] = ll[0], pl[qi][j >> 1][i + 1] = ll[1];
        }
      l[qi] = l[qi] * alpha + ps * exp_scale(-r);
      av[qi] = alpha * vcorr * exp_scale(r - pr[qi]);
      pr[qi] = r;
    }
    const int nk = DIAG && jd == 0 ? 1 : 2;  // 32-key groups with anything unmasked
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      floatx4 u[2] = {zero, zero};
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        if (DIAG && kk >= nk) continue;
        const char* p = vs + granule128(16 * d + l16, 4 * kk + g);
        const half8 vh = *reinterpret_cast<const half8*>(p), vl = *reinterpret_cast<const half8*>(p + G::VPLANE);
#pragma unroll
        for (int qi = 0; qi < 2; ++qi) u[qi] = mfma_f16(vl, ph[qi][kk], u[qi]);
#pragma unroll
        for (int qi = 0; qi < 2; ++qi) u[qi] = mfma_f16(vh, pl[qi][kk], u[qi]);
#pragma unroll
        for (int qi = 0; qi < 2; ++qi) u[qi] = mfma_f16(vh, ph[qi][kk], u[qi]);
      }
#pragma unroll
      for (int qi = 0; qi < 2; ++qi)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[qi][d][e] = __builtin_fmaf(acc[qi][d][e], av[qi], u[qi][e]);
    }
  };

  const int last = min(qb * QB + QB - 1, a.T - 1);  // the block's last query
  const int nkt = last / 64 + 1;
  load(0);
  for (int kt = 0; kt < nkt; ++kt) {
    const int k0 = kt * 64;
    float mk = 0.f, mv = 0.f;
#pragma unroll
    for (int i = 0; i < KS; ++i)
#pragma unroll
      for (int e = 0; e < 8; e += 2) mk = fmaxf(fmaxf(mk, fabsf(kx[i][e])), fabsf(kx[i][e + 1]));
#pragma unroll
    for (int e = 0; e < 8; ++e) mv = fmaxf(fmaxf(mv, fabsf(vx[0][e])), fabsf(vx[1][e]));
    mk = wave_max(mk);
    mv = wave_max(mv);
    if (lane == 0) red[0][w] = mk, red[1][w] = mv;
    __syncthreads();  // the maxima are there, and every wave is done with the previous tile
    mk = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    mv = fmaxf(fmaxf(red[1][0], red[1][1]), fmaxf(red[1][2], red[1][3]));
    const int pk = score_exp(mk), pv_new = min(pv, value_exp(mv));
    again |= mk == INFINITY || mv == INFINITY || pk + pq_min < 16;
    const float sk = kr & 1 ? -exp_scale(pk) : exp_scale(pk), sv = exp_scale(pv_new);
    pv = pv_new;
    // V grown beyond what P's scale can follow
    if (mv > 0.f) pv_top = max(pv_top, pv);
    again |= pv_top - pv > kPExpMax;
    half2v vh[2][4];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int e = 0; e < 8; e += 2) vh[r][e / 2] = split_high(vx[r][e], vx[r][e + 1], r ? -sv : sv, r ? -sv : sv);
    if (__any((DH == 64 || v_live) && out_of_range(__builtin_elementwise_max(high_range(vh[0]), high_range(vh[1]))))) {
      int n = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) n += count_fine(vx[0][i], sv) + count_fine(vx[1][i], sv);
      if (n >= G::FINE && k0 + 64 > a.T) {  // the keys past the last one are copies of it
        n = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const bool in = k0 + 32 * (vg >> 2) + 4 * (vg & 3) + 16 * (i >> 2) + (i & 3) < a.T;
          n += count_fine(vx[0][i], sv, in) + count_fine(vx[1][i], sv, in);
        }
      }
      if (n >= G::FINE) wide = 1;
    }
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      half8 hh, ll;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        half2v h2, l2;
        split2(kx[i][e], kx[i][e + 1], sk, sk, h2, l2);
        hh[e] = h2[0], hh[e + 1] = h2[1];
        ll[e] = l2[0], ll[e + 1] = l2[1];
      }
      char* p = ks + k_granule<G::KROW>(kr, (tid & 3) + 4 * i);
      *reinterpret_cast<half8*>(p) = hh;
      *reinterpret_cast<half8*>(p + G::KPLANE) = ll;
    }
    if (DH == 64 || v_on) {
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        half8 hh, ll;
        const float s = r ? -sv : sv;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const half2v h2 = vh[r][e / 2], l2 = split_low(vx[r][e], vx[r][e + 1], s, s, h2);
          hh[e] = h2[0], hh[e + 1] = h2[1];
          ll[e] = l2[0], ll[e + 1] = l2[1];
        }
        char* p = vs + granule128(2 * vp + r, vg);
        *reinterpret_cast<half8*>(p) = hh;
        *reinterpret_cast<half8*>(p + G::VPLANE) = ll;
      }
    }
    __syncthreads();
    if (kt + 1 < nkt) load(k0 + 64);
    if (k0 <= q0 + 31) {
      const float vcorr = exp_scale(max(pv - pva, -126));
      pva = pv;
      if (k0 + 63 < q0)
        compute(k0, pk, vcorr, std::false_type{});
      else
        compute(k0, pk, vcorr, std::true_type{});
    }
  }

#pragma unroll
  for (int qi = 0; qi < 2; ++qi) {
    const int qrow = q0 + 16 * qi + l16;
    const float ls = rows4_sum(l[qi]);
    const float inv = ls > 0.f ? 1.f / (kPScale * ls) : 0.f;
    bool bad = !(ls - ls == 0.f);
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float o = ldexpf(acc[qi][d][e] * (e & 1 ? -inv : inv), -(pva + pr[qi]));
        acc[qi][d][e] = o;
        bad |= !(o - o == 0.f);
      }
    if (again || wide || __any(bad)) {
      fwd_fp32_rows<DH>(a, Qb, Kb, Vb, row_base, b, h, q0 + 16 * qi, g, l16);
    } else if (qrow < a.T) {
      float* orow = a.out + (row_base + qrow) * a.ld_o + h * DH;
#pragma unroll
      for (int d = 0; d < DT; ++d)
        if (DH % 16 == 0 || 16 * d + 4 * g < DH) *reinterpret_cast<floatx4*>(orow + 16 * d + 4 * g) = acc[qi][d];
      if (g == 0) a.lse[((size_t)b * a.H + h) * a.T + qrow] = (m[qi] + __log2f(ls)) * (1.f / LOG2E);
    }
  }
}

template <int DH>
void launch(const AttnArgs& a, int b, hipStream_t st) {
  hipLaunchKernelGGL(mha_fwd_split_kernel<DH>, dim3(a.H, b, (a.T + QB - 1) / QB), dim3(256), 0, st, a);
}

}  // namespace

namespace aurattn {

void fwd_split(const AttnArgs& a, int b, int d_head, hipStream_t st) {
  switch (d_head) {
    case 8: launch<8>(a, b, st); break;
    case 16: launch<16>(a, b, st); break;
    case 24: launch<24>(a, b, st); break;
    case 32: launch<32>(a, b, st); break;
    case 40: launch<40>(a, b, st); break;
    case 48: launch<48>(a, b, st); break;
    case 56: launch<56>(a, b, st); break;
    default: launch<64>(a, b, st); break;
  }
}

}  // namespace aurattn
