// fp32 GEMM on the fp16 matrix cores: every fp32 operand value is split into
// two fp16 numbers and the products are summed in fp32 by
// v_mfma_f32_16x16x32_f16 (1.8 PFLOP/s with random operands in registers on
// MI355X, where power sets the clock, against 0.15 for the fp32 MFMA).
//
//   x·2^p = h + l,  h = fp16(x·2^p),  l = fp16(x·2^p − h)
//   a·b·2^(pa+pb) ≈ ha·hb + ha·lb + la·hb        (three MFMAs)
//
// h and l hold 23 of the 24 significant bits of x (the last one is lost for
// one value in four) and the dropped la·lb is below 2^-22 of the product, both
// with random sign, while an MFMA rounds once per 32 products where the fp32
// MFMA rounds at each.  The three products of 32 k are summed from zero, small
// ones first, and the sum is added to the accumulator by the VALU: added to
// the accumulator one by one, products far below its last bit would be lost
// the same way in every row (with one large term in each row, as in a softmax
// gradient, that made column sums of the result three times less accurate than
// the fp32 MFMA's).  The MFMA truncates downwards, so odd rows and odd columns
// are scaled by −2^p: the sign of that error alternates over the result.
// Relative error against float64 on normal operands, fp32 MFMA → here: 1.4e-7
// → 0.93e-7 at K = 64, 4.0e-7 → 1.2e-7 at 512, 1.16e-6 → 2.4e-7 at 4096,
// 2.3e-6 → 4.4e-7 at 16384; the same order holds for uniform, all-positive
// and softmax-gradient operands; what is computed again in fp32 (below) has the fp32
// MFMA's error.
//
// fp16 spans only 2^-24 … 2^16, so every row of A and column of B carries its
// own power-of-two scale 2^p.  It starts from the row's first 32 values (their
// largest magnitude goes to 2^13 … 2^14, at least 4 times below the limit) and
// shrinks when a later value would pass the limit; the accumulators of that row
// are then rescaled before the next product is added.
//
// A value below 2^-2 at that scale has an absolute error of up to 2^-25 there
// instead of a relative one, which shows where the row's large values meet zeros or
// small values of the column.  Down to 2^-4 that is 2^-21 of the value.  The values
// below, 2^17 … 2^20 below the row's largest, are counted per row and column (n and
// m): what they can do to a result is at most E = (n + m)·2^-25·2^16.  It stands if E is
// below 2^-21 of the sum of the products' magnitudes, for which there are two
// lower bounds: the result's own magnitude, and, where the first 32 values of row
// and column hold D and D' of 2^9 or more, (D + D' − 32)·2^18, less by the bits that
// the scales were lowered.  (That clears N(0, 1) operands, halves of zeros and GELU
// outputs without a look at the results.)  The others are computed again in fp32: a few of a wave as dot
// products, from more on the block's tile with the fp32 MFMA.  So is a tile with a
// result that is not finite — an infinity or NaN among the operands, or a product
// that overflows —, so that infinities and NaN come out as they do there.
//
// What bounds it: per 32 of K a wave of the 256×256 tile (128×64 outputs)
// issues 96 MFMAs (1536 matrix-core cycles), 128 additions, ≈ 150 operations
// of splitting and checking, 24 fragment reads and 8 LDS writes, and the waves of a
// SIMD hardly overlap the two (matrix cores busy 53 % of the cycles).
// Measured (fp32 MFMA kernels → here): A·B 16384×1024×4096 982 → 376 µs (365
// TFLOP/s), 8192×2048×512 129 → 59 µs, dW 4096×1024 over 16384 rows 1016 →
// 422 µs, 777×1023×513 24.3 → 14.9 µs.  Counting the small values is 2 µs of the
// second and 1.3 of the last (one wave per SIMD there).  Tiles that are computed
// again add the fp32 MFMA's time: 4096×1024×4096 140 µs, all of it again (an outlier
// of 2^12 or more in a row, met by zeros) 370 to 440, where the fp32 kernels take 255.
// The 256×256 tile needs the fewest LDS and L2 bytes per product; the
// smaller tiles serve shapes with few output tiles (choose_plan in gemm.hip).
#include "common.hpp"
#include "gemm_tile.hpp"
#include "gemm_split.hpp"
#include "split16.hpp"

#include <type_traits>

using namespace aurgemm;
using namespace aursplit;

namespace {

// Global vectors of any 4-byte alignment (one load instruction all the same).
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float floatx2u __attribute__((ext_vector_type(2), aligned(4)));

// Scale exponent p of a row whose largest magnitude is m (0 when there is none
// yet), and that of the factor 2^p.
constexpr float kFineBound = 4096.f;    // |result| ≥ this · (n + m), at the scales: E ≤ 2^-21 of it
constexpr int kDenseBound = 64;         // n + m ≤ this · (D + D' − 32): E ≤ 2^-21 of that bound (scales not lowered)
constexpr int kZeroExp = 127;           // of a row of zeros so far, and of no other (but for values below 2^-111)
__device__ __forceinline__ int row_exp(float m) {
  return m == 0.f ? kZeroExp : min(140 - (int)(__float_as_uint(m) >> 23), 126);
}
__device__ __forceinline__ int scale_exp(float s) { return (int)((__float_as_uint(s) >> 23) & 255) - 127; }

// Byte offset of granule q (4 k) of row r in an fp32 tile [ROWS][32].
__device__ __forceinline__ int fp32_granule(int r, int q) { return r * 128 + ((q ^ r) & 7) * 16; }

// One operand's share of a thread: NO "octets", each 8 consecutive k of one
// row (of A, or column of B) in a stage of 32 k.
//   k-contiguous: octet i is row tid/4 + i·NT/4, k 8·(tid%4) — two float4 loads.
//   k-strided: the thread owns CV neighbouring rows at one k octet per group
//   (a wave covers 16·CV rows × 32 k), eight loads of CV floats, one per k; the
//   transposition is only which registers are packed together.
// A row's four octets sit in the lanes l, l^1, l^2, l^3 (k-contiguous) or
// l, l^16, l^32, l^48 (k-strided), so its scale is kept in registers.
template <int ROWS, int NT, bool KC>
struct SplitOperand {
  static constexpr int NO = ROWS * 4 / NT;
  static constexpr int CV = KC ? 1 : (NO < 2 ? 1 : 2);
  static constexpr int NG = NO / CV;  // load groups
  static_assert(NO >= 1 && NO % CV == 0 && ROWS % (16 * CV) == 0, "tile/threads mismatch");
  const float* base;  // tile row 0 at the k of the next stage to load
  int ld, koct;       // koct: first k of the thread's octets within a stage
  unsigned off[NG];   // byte offset of the group from base (32 bits: ld < 2^21)
  int shift[NG];      // k-strided: rows the vector was moved back to stay inside the operand
  int row0;           // row of octet 0; octet o is step(o) rows further
  unsigned lds;       // its byte offset in an LDS plane
  float x[NO][8], s[NO];
  __device__ static constexpr int step(int o) { return KC ? o * (NT / 4) : (o / CV) * (NT / 4) * CV + o % CV; }

  __device__ __forceinline__ void init(const float* X, int ld_, int r0, int rows, int k0, int tid) {
    ld = ld_;
    if constexpr (KC) {
      koct = 8 * (tid & 3);
      base = X + (size_t)r0 * ld + k0;
      row0 = tid >> 2;
      // a row past the operand reads its last row: its results are not stored
#pragma unroll
      for (int i = 0; i < NO; ++i)
        off[i] = ((unsigned)min(row0 + step(i), rows - 1 - r0) * (unsigned)ld + koct) * 4u;
    } else {
      const int lane = tid & 63, wave = tid >> 6;
      koct = 8 * (lane >> 4);
      // One row before the tile, so that the offset of a pair moved back over
      // the tile's first row (cl = −1: the tile has a single row, the operand
      // at least two) stays positive.
      base = X + (ptrdiff_t)k0 * ld + r0 - 1;
      row0 = wave * 16 * CV + CV * (lane & 15);
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const int c = row0 + step(i * CV), cl = min(c, rows - r0 - CV);
        shift[i] = c - cl;
        off[i] = ((unsigned)koct * (unsigned)ld + (unsigned)(cl + 1)) * 4u;
      }
    }
    lds = split_granule(row0, koct >> 3);
  }
  __device__ __forceinline__ static const float* at(const float* b, unsigned bytes) {
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(b) + bytes);
  }
  // Group i of the stage at `base`; GUARD: only the first kr k exist.
  template <bool GUARD>
  __device__ __forceinline__ void load(int i, int kr) {
    if constexpr (KC) {
      if constexpr (!GUARD) {
        const floatx4u a = *reinterpret_cast<const floatx4u*>(at(base, off[i]));
        const floatx4u b = *reinterpret_cast<const floatx4u*>(at(base + 4, off[i]));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[i][e] = a[e], x[i][4 + e] = b[e];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[i][e] = koct + e < kr ? at(base, off[i])[e] : 0.f;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float* p = at(base + (size_t)e * ld, off[i]);
        if constexpr (CV == 1) {
          x[i][e] = !GUARD || koct + e < kr ? p[0] : 0.f;
        } else {
          floatx2u v = {0.f, 0.f};
          if (!GUARD || koct + e < kr) v = *reinterpret_cast<const floatx2u*>(p);
          x[2 * i][e] = v[0];
          x[2 * i + 1][e] = v[1];
        }
      }
    }
  }
  template <bool GUARD>
  __device__ __forceinline__ void load_all(int kr) {
#pragma unroll
    for (int i = 0; i < NG; ++i) load<GUARD>(i, kr);
  }
  __device__ __forceinline__ void advance() { base += KC ? (size_t)32 : (size_t)32 * ld; }

  __device__ __forceinline__ float octet_max(int o) const {
    float m = fmaxf(fabsf(x[o][0]), fabsf(x[o][1]));
#pragma unroll
    for (int e = 2; e < 8; e += 2) m = fmaxf(fmaxf(m, fabsf(x[o][e])), fabsf(x[o][e + 1]));
    return m;
  }
  // Values of octet o that are too small for the row's scale; zeros are exact.
  __device__ __forceinline__ int octet_fine(int o) const {
    int n = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) n += (x[o][e] != 0.f) & (fabsf(x[o][e] * s[o]) < kSplitFine);
    return n;
  }
  __device__ __forceinline__ int octet_from(int o, float least) const {
    int n = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) n += fabsf(x[o][e]) >= least;
    return n;
  }
  // Over a row's four octets (quad permutes, or row and half swaps).
  template <class Op>
  __device__ __forceinline__ static int over_row(int v, Op op) {
    if constexpr (KC) {
      v = op(v, __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true));
      return op(v, __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true));
    } else {
      const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
      v = op(s[0], s[1]);
      const auto t = __builtin_amdgcn_permlane32_swap(v, v, false, false);
      return op(t[0], t[1]);
    }
  }
  __device__ __forceinline__ static int row_sum(int n) {
    return over_row(n, [](int a, int b) { return a + b; });
  }
  __device__ __forceinline__ static float row_max(float m) {
    return __int_as_float(over_row(__float_as_int(m), [](int a, int b) {
      return __float_as_int(fmaxf(__int_as_float(a), __int_as_float(b)));
    }));
  }
  // Odd rows are scaled by −2^p (see the head of the file).
  __device__ __forceinline__ void set_exp(int o, int p) {
    s[o] = exp_scale(p);
    if ((row0 + step(o)) & 1) s[o] = -s[o];
  }
  // k-strided rows whose vector was moved back by one hold their value in the
  // second component (the last row of an odd extent)
  __device__ __forceinline__ void align(int o) {
    if constexpr (!KC && CV == 2) {
      if (o % 2 == 0 && shift[o / 2]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[o][e] = x[o + 1][e];
      }
    }
  }
  // The high parts of octet o.
  __device__ __forceinline__ void high(int o, half2v (&h)[4]) const {
#pragma unroll
    for (int e = 0; e < 8; e += 2) h[e / 2] = split_high(x[o][e], x[o][e + 1], s[o], s[o]);
  }
  // h and l of octet o as two 16-byte granules of the LDS planes [ROWS][32].
  __device__ __forceinline__ void store(int o, const half2v (&hh)[4], char* planes) const {
    half8 h, l;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const half2v ll = split_low(x[o][e], x[o][e + 1], s[o], s[o], hh[e / 2]);
      h[e] = hh[e / 2][0], h[e + 1] = hh[e / 2][1];
      l[e] = ll[0], l[e + 1] = ll[1];
    }
    char* p = planes + lds + step(o) * 64;
    *reinterpret_cast<half8*>(p) = h;
    *reinterpret_cast<half8*>(p + ROWS * 64) = l;
  }
  // The octets' values as they are, [ROWS][32] floats.
  __device__ __forceinline__ void store_fp32(char* tile) const {
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      const int r = row0 + step(o), q = koct >> 2;
      *reinterpret_cast<floatx4*>(tile + fp32_granule(r, q)) = floatx4{x[o][0], x[o][1], x[o][2], x[o][3]};
      *reinterpret_cast<floatx4*>(tile + fp32_granule(r, q + 1)) = floatx4{x[o][4], x[o][5], x[o][6], x[o][7]};
    }
  }
};

// Result (r, c) again in fp32, by the whole wave.
template <bool AK, bool BKC>
__device__ __forceinline__ float fp32_dot(const GemmArgs& g, int r, int c, int kbeg, int kend, int lane) {
  const size_t sa = AK ? 1 : g.lda, sb = BKC ? 1 : g.ldb;
  const float* pa = g.A + (size_t)r * (AK ? g.lda : 1);
  const float* pb = g.B + (size_t)c * (BKC ? g.ldb : 1);
  constexpr int U = 8;
  float sum[U] = {};
#pragma unroll 1
  for (int k0 = kbeg + lane; k0 < kend; k0 += 64 * U)
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int k = k0 + 64 * i;
      if (k < kend) sum[i] = __builtin_fmaf(pa[k * sa], pb[k * sb], sum[i]);
    }
  float v = ((sum[0] + sum[1]) + (sum[2] + sum[3])) + ((sum[4] + sum[5]) + (sum[6] + sum[7]));
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// acc += u, at this place: left alone the compiler moves the additions to the
// end of the stage and keeps every u alive until then.
__device__ __forceinline__ void add_here(floatx4& acc, floatx4 u) {
  acc += u;
  asm volatile("" : "+v"(acc));
}

template <int BM, int BN, int WGM, int WGN, bool AK, bool BKC, bool LATE>
__global__ void __launch_bounds__(64 * WGM * WGN, BM == 64 ? 4 : 2) gemm_f16x3(GemmArgs g) {
  select_batch(g);
  constexpr int NT = 64 * WGM * WGN;
  constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
  constexpr int STAGE = (BM + BN) * 128;  // bytes: h and l planes of both operands
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];
  // Rescaling notes, one per row of A and column of B and stage parity: (stage,
  // change of the exponent); flag[parity] = the stage that has any.
  __shared__ int2 note[2][BM + BN];
  __shared__ int flag[2];
  // Of each row of A and column of B: the values too small for their scale; those
  // of the first 32 that are large at the first scale, and 256 times its exponent
  __shared__ int fine[BM + BN], dense[BM + BN];
  __shared__ int rough;  // a result may have to be looked at
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WGN, wn = wave % WGN;
  const int g16 = lane >> 4, l16 = lane & 15;
  // Tile order: a contiguous run of tiles per XCD, walked in groups of 8 tile
  // rows, as the fp32 kernels.
  constexpr int GM = 8;
  const int ntiles = g.tiles_m * g.tiles_n;
  int pid = blockIdx.x;
  if ((ntiles & 7) == 0) pid = (pid & 7) * (ntiles >> 3) + (pid >> 3);
  const int per_group = GM * g.tiles_n;
  const int first_m = (pid / per_group) * GM;
  const int gsz = min(g.tiles_m - first_m, GM);
  const int m0 = (first_m + (pid % per_group) % gsz) * BM, n0 = ((pid % per_group) / gsz) * BN;
  const int kbeg = blockIdx.z * g.k_chunk;
  const int kend = min(g.K, kbeg + g.k_chunk);
  const int nk = (kend - kbeg + 31) / 32;
  const int ktail = (kend - kbeg) & 31;  // k of a partial last stage

  SplitOperand<BM, NT, AK> la;
  SplitOperand<BN, NT, BKC> lb;
  constexpr int NOA = decltype(la)::NO, NOB = decltype(lb)::NO, NO = NOA + NOB;
  la.init(g.A, g.lda, m0, g.M, kbeg, tid);
  lb.init(g.B, g.ldb, n0, g.N, kbeg, tid);

  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  if (nk == 1 && ktail) {
    la.template load_all<true>(ktail);
    lb.template load_all<true>(ktail);
  } else {
    la.template load_all<false>(0);
    lb.template load_all<false>(0);
  }
  for (int i = tid; i < 2 * (BM + BN); i += NT) (&note[0][0])[i] = int2{-1, 0};
  if (tid < 2) flag[tid] = -1;
  if (tid == 0) rough = 0;
  auto first = [&](auto& op, int o, int note0, char* planes) {
    op.align(o);
    const int p = row_exp(op.row_max(op.octet_max(o))), row = note0 + op.row0 + op.step(o);
    op.set_exp(o, p);
    half2v h[4];
    op.high(o, h);
    op.store(o, h, planes);
    int n = op.octet_from(o, exp_scale(9 - p));
    if (__any(out_of_range(high_range(h)))) n |= op.octet_fine(o) << 8;
    n = op.row_sum(n);
    if (op.koct == 0) {
      fine[row] = n >> 8;
      dense[row] = 256 * p + (n & 255);
    }
  };
#pragma unroll
  for (int o = 0; o < NOA; ++o) first(la, o, 0, smem);
#pragma unroll
  for (int o = 0; o < NOB; ++o) first(lb, o, BM, smem + BM * 128);
  la.advance();
  lb.advance();
  if (nk > 1) {
    if (nk == 2 && ktail) {
      la.template load_all<true>(ktail);
      if (!LATE) lb.template load_all<true>(ktail);
    } else {
      la.template load_all<false>(0);
      if (!LATE) lb.template load_all<false>(0);
    }
    la.advance();
    if (!LATE) lb.advance();
  }
  __syncthreads();

  // Octets of stage kt + 1 with values out of range.  A row that passes the limit is
  // rescaled; values too small for its scale are counted.  What the sums hold may
  // underflow by a scale 2^60 below the first: that counts as one value.
  auto rescale = [&](auto& op, int o, int kt, int note0) {
    const float rm = op.row_max(op.octet_max(o));
    if (rm * fabsf(op.s[o]) > kSplitLimit) {
      const int row = note0 + op.row0 + op.step(o), p = row_exp(rm), old = scale_exp(op.s[o]);
      note[(kt + 1) & 1][row] = int2{kt + 1, p - old};
      flag[(kt + 1) & 1] = kt + 1;
      if (op.koct == 0) {
        if (old == kZeroExp)
          dense[row] = 256 * p;
        else if (p < (dense[row] >> 8) - 60)
          atomicAdd(&fine[row], 1);
      }
      op.set_exp(o, p);
    }
  };
  auto count = [&](auto& op, int o, int note0) {
    const int n = op.octet_fine(o);
    if (n) atomicAdd(&fine[note0 + op.row0 + op.step(o)], n);
  };
  half2v hh[NO][4];  // high parts of the octets to be split next
  auto high = [&](int o) {
    if (o < NOA)
      la.high(o, hh[o]);
    else
      lb.high(o - NOA, hh[o]);
  };
  ushort2v range;  // of them
  auto high_octets = [&](int o0, int o1) {
#pragma unroll
    for (int o = o0; o < o1; ++o) {
      if (o < NOA)
        la.align(o);
      else
        lb.align(o - NOA);
      high(o);
      range = o == o0 ? high_range(hh[o]) : __builtin_elementwise_max(range, high_range(hh[o]));
    }
  };
  auto check_octets = [&](int o0, int o1, int kt) {
    if (__any(out_of_range(range))) {
#pragma unroll
      for (int o = o0; o < o1; ++o) {
        const float m = o < NOA ? la.octet_max(o) * fabsf(la.s[o]) : lb.octet_max(o - NOA) * fabsf(lb.s[o - NOA]);
        if (__any(m > kSplitLimit)) {
          if (o < NOA)
            rescale(la, o, kt, 0);
          else
            rescale(lb, o - NOA, kt, BM);
          high(o);
        }
        if (o < NOA)
          count(la, o, 0);
        else
          count(lb, o - NOA, BM);
      }
    }
  };
  // MFMA operands of 16 rows: lane group g holds the k octet g of row l16.
  half8 ah, al, bh[TN], bl[TN];
  const int fa = split_granule(l16, g16) + wm * WM * 64, fb = split_granule(l16, g16) + BM * 128 + wn * WN * 64;
  auto read_a = [&](const char* st, int i) {
    ah = *reinterpret_cast<const half8*>(st + fa + i * 1024);
    al = *reinterpret_cast<const half8*>(st + fa + i * 1024 + BM * 64);
  };
  auto read_b = [&](const char* st, int j) {
    bh[j] = *reinterpret_cast<const half8*>(st + fb + j * 1024);
    bl[j] = *reinterpret_cast<const half8*>(st + fb + j * 1024 + BN * 64);
  };
  read_a(smem, 0);
#pragma unroll
  for (int j = 0; j < TN; ++j) read_b(smem, j);
  // LATE (the 256×256 tile, whose 256 registers per wave are full): the
  // registers hold one operand of the next stage at a time, each loaded half a
  // stage ahead; the other tiles load both a whole stage ahead.
  // One stage, in TM steps of 16 rows.  Every step but the last reads the next
  // step's A fragments, runs its 3·TN MFMAs and, spread among them, splits one
  // octet of stage kt + 1 into the other LDS stage and reloads its registers.
  // The barrier stands before the last step: by then the wave has read all it
  // needs of the stage and written its share of the next one, so the last
  // step's MFMAs cover the first fragment reads of the next stage (a column's
  // fragments are replaced as soon as their last MFMA is issued).
  // An octet's high parts and their range are found under the products of the step
  // before it by the LATE tile (dx 16384×1024×4096: 390 → 378 µs), at the start of
  // its own by the others (their registers are loaded too shortly before: 15.6 →
  // 16.7 µs at 777×1023×513).
  constexpr int S = TM > 1 ? TM - 1 : 1;  // steps that convert
  // octets [first_octet(i), first_octet(i + 1)) are split in step i
  constexpr auto first_octet = [](int i) {
    if (!LATE) return i * NO / S;
    return i <= 2 ? 0 : i <= 6 ? NOA : NO;
  };
  // MODE 0: stage kt + 2 is loaded whole; 1: it is the partial last one; 2:
  // there is none; 3: the last stage, nothing to convert.
  auto step = [&](int kt, auto mode) {
    constexpr int MODE = decltype(mode)::value;
    const char* sa = smem + (kt & 1) * STAGE;
    char* na = smem + ((kt + 1) & 1) * STAGE;
    char* nb = na + BM * 128;
    if (flag[kt & 1] == kt) {
      int dc[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int2 v = note[kt & 1][BM + wn * WN + 16 * j + l16];
        dc[j] = v.x == kt ? v.y : 0;
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int2 v = note[kt & 1][wm * WM + 16 * i + 4 * g16 + e];
          const int dr = v.x == kt ? v.y : 0;
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j][e] = ldexpf(acc[i][j][e], dr + dc[j]);
        }
    }
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    constexpr int JB = TN > 1 ? 2 : 1;  // columns in flight
    floatx4 u[2][JB];                   // products of the current and the previous pair
    // The pair (i, j0)'s products, and the previous pair's addition under them.
    auto pair = [&](int i, int j0, const half8& ph, const half8& pl) {
      const int q = (i * (TN / JB) + j0 / JB) & 1;
#pragma unroll
      for (int j = 0; j < JB; ++j) u[q][j] = mfma_f16(pl, bh[j0 + j], zero);
#pragma unroll
      for (int j = 0; j < JB; ++j) u[q][j] = mfma_f16(ph, bl[j0 + j], u[q][j]);
#pragma unroll
      for (int j = 0; j < JB; ++j) u[q][j] = mfma_f16(ph, bh[j0 + j], u[q][j]);
      const int i1 = j0 ? i : i - 1, j1 = j0 ? j0 - JB : TN - JB;
      if (i1 >= 0) {
#pragma unroll
        for (int j = 0; j < JB; ++j) add_here(acc[i1][j1 + j], u[q ^ 1][j]);
      }
    };
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const half8 ch = ah, cl = al;
      if (i + 1 < TM) {
        const int o0 = MODE == 3 ? 0 : first_octet(i), o1 = MODE == 3 ? 0 : first_octet(i + 1);
        if (!LATE) high_octets(o0, o1);
        if (o1 > o0) check_octets(o0, o1, kt);
        read_a(sa, i + 1);
#pragma unroll
        for (int j0 = 0; j0 < TN; j0 += JB) pair(i, j0, ch, cl);
#pragma unroll
        for (int o = o0; o < o1; ++o) {
          if (o < NOA) {
            la.store(o, hh[o], na);
            if ((o + 1) % la.CV == 0 && MODE < 2 && !LATE) la.template load<MODE == 1>(o / la.CV, ktail);
            if (LATE && o + 1 == NOA) {  // B of stage kt + 1 takes A's registers
              if (MODE == 2 && ktail)
                lb.template load_all<true>(ktail);
              else
                lb.template load_all<false>(0);
              lb.advance();
            }
          } else {
            lb.store(o - NOA, hh[o], nb);
            if ((o - NOA + 1) % lb.CV == 0 && MODE < 2 && !LATE) lb.template load<MODE == 1>((o - NOA) / lb.CV, ktail);
            if (LATE && o + 1 == NO && MODE < 2) la.template load_all<MODE == 1>(ktail);  // A of stage kt + 2
          }
        }
        if (LATE && MODE < 3 && i + 2 < TM) high_octets(first_octet(i + 1), first_octet(i + 2));
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int r = 0; r < 3 * TN; ++r) {
          constexpr int per = LATE ? 2 : (NO + S - 1) / S;
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (o1 > o0)
            __builtin_amdgcn_sched_group_barrier(0x002, 2 + 2 * per, 0);
          else
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      } else {
        if constexpr (MODE < 3) {
          __syncthreads();
          read_a(na, 0);
        }
#pragma unroll
        for (int j0 = 0; j0 < TN; j0 += JB) {
          pair(i, j0, ch, cl);
          if constexpr (MODE < 3) {
#pragma unroll
            for (int j = j0; j < j0 + JB; ++j) read_b(na, j);
          }
        }
#pragma unroll
        for (int j = 0; j < JB; ++j) add_here(acc[i][TN - JB + j], u[(TM * (TN / JB) - 1) & 1][j]);
      }
    }
    if constexpr (MODE < 2) {
      la.advance();
      if (!LATE) lb.advance();
    }
  };
  int kt = 0;
  for (; kt + 2 < nk - (ktail ? 1 : 0); ++kt) step(kt, std::integral_constant<int, 0>{});
  if (kt + 2 < nk) step(kt++, std::integral_constant<int, 1>{});
  if (kt + 1 < nk) step(kt++, std::integral_constant<int, 2>{});
  step(kt, std::integral_constant<int, 3>{});

  // The rows' and columns' final exponents, through the notes' memory.
  __syncthreads();
  int* ex = reinterpret_cast<int*>(&note[0][0]);
  // The large values of a row and a column clear their result if n + m ≤
  // 64·(D + D' − 32)·2^-(d + d'), with d the bits by which a scale was lowered; so they
  // do if n ≤ 8·(D − 16)·2^-d and d ≤ 3 for both.  dense becomes D + 256·d.  Rows
  // that are zero or past the operand are never in doubt.
  constexpr int kNever = -(1 << 30);
  auto last = [&](auto& op, int o, int note0, int rows) {
    const int r = op.row0 + op.step(o), row = note0 + r;
    if (op.koct == 0) {
      const int p = scale_exp(op.s[o]), big = dense[row] & 255, d = min((dense[row] >> 8) - p, 15);
      ex[row] = p;
      dense[row] = big + 256 * d;
      if (p == kZeroExp || r >= rows)
        fine[row] = kNever;
      else if (d > 3 || fine[row] > (kDenseBound / 8 * (big - 16)) >> d)
        rough = 1;
    }
  };
#pragma unroll
  for (int o = 0; o < NOA; ++o) last(la, o, 0, g.M - m0);
#pragma unroll
  for (int o = 0; o < NOB; ++o) last(lb, o, BM, g.N - n0);
  __syncthreads();
  int pc[TN];
  // Results to compute again: bit 4j + e of fl[i].
  unsigned fl[TM], worst = 0;
  int nfl = 0;
  if (rough) {
    int nc[TN], wc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      nc[j] = fine[BM + wn * WN + 16 * j + l16];
      wc[j] = dense[BM + wn * WN + 16 * j + l16];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      fl[i] = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = wm * WM + 16 * i + 4 * g16 + e, nr = fine[row], wr = dense[row];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int n = nr + nc[j], w = wr + wc[j], most = (kDenseBound * max((w & 255) - 32, 0)) >> (w >> 8);
          const float bound = n > most ? kFineBound * (float)n : 0.f;
          fl[i] |= (fabsf(acc[i][j][e]) < bound ? 1u : 0u) << (4 * j + e);
        }
      }
      nfl += __popc(fl[i]);
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) nfl += __shfl_xor(nfl, m, 64);
  }
  const unsigned odd = (unsigned)l16 << 31;
#pragma unroll
  for (int j = 0; j < TN; ++j) pc[j] = ex[BM + wn * WN + 16 * j + l16];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int pr = ex[wm * WM + 16 * i + 4 * g16 + e];
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        // rows and columns of different parity carry a minus sign
        const float v = __uint_as_float(__float_as_uint(ldexpf(acc[i][j][e], -(pr + pc[j]))) ^ (odd ^ (unsigned)(e & 1) << 31));
        acc[i][j][e] = v;
        worst = max(worst, __float_as_uint(v) & 0x7fffffffu);
      }
    }
  }
  const int r0 = m0 + wm * WM, c0 = n0 + wn * WN;
  // One result as a dot product takes the wave 2 µs (K = 4096, contiguous operands)
  // to 5 µs (strided).
  constexpr int kDots = AK && BKC ? 32 : 8;
  if (nfl > kDots || __any(worst >= 0x7f800000u)) rough = 2;
  __syncthreads();
  if (rough == 2) {
    // The block's tile with the fp32 MFMA: 32 k at a time through LDS as they are,
    // the next ones loaded under the products.  (k-groups of 16: lane group g holds
    // the k 4g … 4g + 3 of each.)
    auto load = [&](int kt) {
      if (kt + 1 == nk && ktail) {
        la.template load_all<true>(ktail);
        lb.template load_all<true>(ktail);
      } else {
        la.template load_all<false>(0);
        lb.template load_all<false>(0);
      }
      la.advance();
      lb.advance();
    };
    la.init(g.A, g.lda, m0, g.M, kbeg, tid);
    lb.init(g.B, g.ldb, n0, g.N, kbeg, tid);
    load(0);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt) {
      char* st = smem + (kt & 1) * STAGE;
#pragma unroll
      for (int o = 0; o < NOA; ++o) la.align(o);
#pragma unroll
      for (int o = 0; o < NOB; ++o) lb.align(o);
      la.store_fp32(st);
      lb.store_fp32(st + BM * 128);
      __syncthreads();
      if (kt + 1 < nk) load(kt + 1);
#pragma unroll
      for (int q = 0; q < 8; q += 4) {
        floatx4 a, b[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j)
          b[j] = *reinterpret_cast<const floatx4*>(st + BM * 128 + fp32_granule(wn * WN + 16 * j + l16, q + g16));
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          a = *reinterpret_cast<const floatx4*>(st + fp32_granule(wm * WM + 16 * i + l16, q + g16));
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = mfma16x16x4(a[e], b[j][e], acc[i][j]);
        }
      }
    }
    nfl = 0;
  }
  if (nfl == 0) {  // the usual way out
    write_tiles(g, acc, r0, c0, g16, l16, m0 + BM <= g.M && n0 + BN <= g.N);
    return;
  }
  // The masks go to LDS (no wave reads the stages any more) for a loop over strips
  // of 16 rows.
  unsigned short* masks = reinterpret_cast<unsigned short*>(smem) + wave * (TM * 64) + lane;
#pragma unroll
  for (int i = 0; i < TM; ++i) masks[64 * i] = (unsigned short)fl[i];
  write_tiles(g, acc, r0, c0, g16, l16, false, [&](int i, int j, int e) { return fl[i] >> (4 * j + e) & 1; });
#pragma unroll 1
  for (int i = 0; i < TM; ++i) {
    unsigned mine = masks[64 * i];
#pragma unroll 1
    for (unsigned long long who = __ballot(mine); who; who = __ballot(mine)) {
      const int at = __ffsll(who) - 1, q = __ffs(__builtin_amdgcn_readlane(mine, at)) - 1;
      if (lane == at) mine &= mine - 1;
      const int r = r0 + 16 * i + 4 * (at >> 4) + (q & 3), c = c0 + 16 * (q >> 2) + (at & 15);
      const float v = fp32_dot<AK, BKC>(g, r, c, kbeg, kend, lane);
      if (lane == 0) {
        if (g.split)
          g.P[((size_t)blockIdx.z * g.M + r) * g.N + c] = v;
        else
          apply_epilogue(g.epi, g.C, (size_t)r * g.ldc + c, v);
      }
    }
  }
}

template <int BM, int BN, int WGM, int WGN>
void launch(const GemmArgs& a, bool ak, bool bkc, int splits, int batch, hipStream_t st) {
  constexpr bool LATE = BM == 256 && BN == 256;
  const dim3 grid(a.tiles_m * a.tiles_n, batch, splits), block(64 * WGM * WGN);
  if (ak && bkc)
    hipLaunchKernelGGL((gemm_f16x3<BM, BN, WGM, WGN, true, true, LATE>), grid, block, 0, st, a);
  else if (ak)
    hipLaunchKernelGGL((gemm_f16x3<BM, BN, WGM, WGN, true, false, LATE>), grid, block, 0, st, a);
  else if (bkc)
    hipLaunchKernelGGL((gemm_f16x3<BM, BN, WGM, WGN, false, true, LATE>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((gemm_f16x3<BM, BN, WGM, WGN, false, false, LATE>), grid, block, 0, st, a);
}

}  // namespace

namespace aur {

void gemm_split_launch(const GemmArgs& a, int bm, int bn, bool a_kcontig, bool b_kcontig, int splits, int batch,
                       hipStream_t st) {
  if (bm == 256 && bn == 256)
    launch<256, 256, 2, 4>(a, a_kcontig, b_kcontig, splits, batch, st);
  else if (bm == 256)
    launch<256, 128, 4, 2>(a, a_kcontig, b_kcontig, splits, batch, st);
  else if (bm == 128)
    launch<128, 128, 2, 2>(a, a_kcontig, b_kcontig, splits, batch, st);
  else
    launch<64, 64, 2, 2>(a, a_kcontig, b_kcontig, splits, batch, st);
}

}  // namespace aur
