// fp32 GEMM on the fp16 matrix cores: every fp32 operand value is split into
// two fp16 numbers and the products are summed in fp32 by
// v_mfma_f32_16x16x32_f16 (1.9 PFLOP/s with random operands in registers on
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
// 2.3e-6 → 4.4e-7 at 16384; the same order holds for uniform, all-positive,
// softmax-gradient and widely scaled operands.
//
// fp16 spans only 2^-24 … 2^16, so every row of A and column of B carries its
// own power-of-two scale 2^p.  It starts from the row's first 32 values (their
// largest magnitude goes to 2^7 … 2^8, 128 times below the limit) and shrinks
// when a later value would pass 2^15; the accumulators of that row are then
// rescaled (exactly) before the next product is added.  Values far below the
// row's largest lose relative precision only (their absolute error stays under
// 2^-38 of it).  A result that is not finite — an infinity or NaN among the
// operands, or a product that overflows — is recomputed for the wave's whole
// sub-tile with the fp32 MFMA, so infinities and NaN come out as they do there.
//
// What bounds it: per 32 of K a wave of the 256×256 tile (128×64 outputs)
// issues 96 MFMAs (1536 matrix-core cycles), 128 additions, ≈ 130 operations
// of splitting and checking, 24 fragment reads and 8 LDS writes; the matrix
// cores are busy 55 % of the time and power holds the clock at 1.7-1.9 GHz.
// Measured (fp32 MFMA kernels → here): A·Bᵀ 16384×1024×4096 970 → 386 µs (355
// TFLOP/s), 8192×2048×512 129 → 59 µs, dW 4096×1024 over 16384 rows 1016 →
// 437 µs.  The 256×256 tile needs the fewest LDS and L2 bytes per product; the
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

// Scale exponents: p for a row whose first values' largest magnitude is m (0
// when there is none yet), the lowered p for a row that met a larger m, and
// the factor 2^p.
constexpr float kSplitLimit = 32768.f;  // largest scaled magnitude let through
__device__ __forceinline__ int first_exp(float m) { return min(134 - (int)(__float_as_uint(m) >> 23), 127); }
__device__ __forceinline__ int lowered_exp(float m) { return 140 - (int)(__float_as_uint(m) >> 23); }
__device__ __forceinline__ int scale_exp(float s) { return (int)((__float_as_uint(s) >> 23) & 255) - 127; }

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
  __device__ __forceinline__ static float row_max(float m) {
    m = fmaxf(m, __shfl_xor(m, KC ? 1 : 16, 64));
    return fmaxf(m, __shfl_xor(m, KC ? 2 : 32, 64));
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
  // h and l of octet o as two 16-byte granules of the LDS planes [ROWS][32].
  __device__ __forceinline__ void store(int o, char* planes) const {
    half8 h, l;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      half2v hh, ll;
      split2(x[o][e], x[o][e + 1], s[o], s[o], hh, ll);
      h[e] = hh[0], h[e + 1] = hh[1];
      l[e] = ll[0], l[e + 1] = ll[1];
    }
    char* p = planes + lds + step(o) * 64;
    *reinterpret_cast<half8*>(p) = h;
    *reinterpret_cast<half8*>(p + ROWS * 64) = l;
  }
};

// The wave's sub-tile again with the fp32 MFMA, straight from memory: only for
// results that are not finite.
template <int TM, int TN, bool AK, bool BKC>
__device__ __forceinline__ void fp32_tile(const GemmArgs& g, floatx4 (&acc)[TM][TN], int r0, int c0, int kbeg,
                                          int kend, int g16, int l16) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int k0 = kbeg; k0 < kend; k0 += 4) {
    const int k = k0 + g16;
    float a[TM], b[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const size_t r = min(r0 + 16 * i + l16, g.M - 1);
      a[i] = k < kend ? (AK ? g.A[r * g.lda + k] : g.A[(size_t)k * g.lda + r]) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const size_t c = min(c0 + 16 * j + l16, g.N - 1);
      b[j] = k < kend ? (BKC ? g.B[c * g.ldb + k] : g.B[(size_t)k * g.ldb + c]) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mfma16x16x4(a[i], b[j], acc[i][j]);
  }
}

// acc += u, at this place: left alone the compiler moves the additions to the
// end of the stage and keeps every u alive until then.
__device__ __forceinline__ void add_here(floatx4& acc, floatx4 u) {
  acc += u;
  asm volatile("" : "+v"(acc));
}

template <int BM, int BN, int WGM, int WGN, bool AK, bool BKC, bool LATE>
__global__ void __launch_bounds__(64 * WGM * WGN, 2) gemm_f16x3(GemmArgs g) {
  select_batch(g);
  constexpr int NT = 64 * WGM * WGN;
  constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
  constexpr int STAGE = (BM + BN) * 128;  // bytes: h and l planes of both operands
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];
  // Rescaling notes, one per row of A and column of B and stage parity: (stage,
  // change of the exponent); flag[parity] = the stage that has any.
  __shared__ int2 note[2][BM + BN];
  __shared__ int flag[2];
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
#pragma unroll
  for (int o = 0; o < NOA; ++o) {
    la.align(o);
    la.set_exp(o, first_exp(la.row_max(la.octet_max(o))));
    la.store(o, smem);
  }
#pragma unroll
  for (int o = 0; o < NOB; ++o) {
    lb.align(o);
    lb.set_exp(o, first_exp(lb.row_max(lb.octet_max(o))));
    lb.store(o, smem + BM * 128);
  }
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

  // Octet o of stage kt + 1: its row is rescaled if it passes the limit (rare).
  auto check = [&](auto& op, int o, int kt, int note0) {
    op.align(o);
    const float m = op.octet_max(o);
    if (__any(m * fabsf(op.s[o]) > kSplitLimit)) {
      const float rm = op.row_max(m);
      if (rm * fabsf(op.s[o]) > kSplitLimit) {
        const int p = lowered_exp(rm);
        note[(kt + 1) & 1][note0 + op.row0 + op.step(o)] = int2{kt + 1, p - scale_exp(op.s[o])};
        flag[(kt + 1) & 1] = kt + 1;
        op.set_exp(o, p);
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
  // MODE 0: stage kt + 2 is loaded whole; 1: it is the partial last one; 2:
  // there is none; 3: the last stage, nothing to convert.
  auto step = [&](int kt, auto mode) {
    constexpr int MODE = decltype(mode)::value;
    constexpr int S = TM > 1 ? TM - 1 : 1;  // steps that convert
    // octets [first_octet(i), first_octet(i + 1)) are split in step i
    constexpr auto first_octet = [](int i, int m) {
      if (m == 3) return 0;
      if (!LATE) return i * NO / S;
      return i <= 2 ? 0 : i <= 6 ? NOA : NO;
    };
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
        const int o0 = first_octet(i, MODE), o1 = first_octet(i + 1, MODE);
#pragma unroll
        for (int o = o0; o < o1; ++o) {
          if (o < NOA)
            check(la, o, kt, 0);
          else
            check(lb, o - NOA, kt, BM);
        }
        read_a(sa, i + 1);
#pragma unroll
        for (int j0 = 0; j0 < TN; j0 += JB) pair(i, j0, ch, cl);
#pragma unroll
        for (int o = o0; o < o1; ++o) {
          if (o < NOA) {
            la.store(o, na);
            if ((o + 1) % la.CV == 0 && MODE < 2 && !LATE) la.template load<MODE == 1>(o / la.CV, ktail);
            if (LATE && o + 1 == NOA) {  // B of stage kt + 1 takes A's registers
              if (MODE == 2 && ktail)
                lb.template load_all<true>(ktail);
              else
                lb.template load_all<false>(0);
              lb.advance();
            }
          } else {
            lb.store(o - NOA, nb);
            if ((o - NOA + 1) % lb.CV == 0 && MODE < 2 && !LATE) lb.template load<MODE == 1>((o - NOA) / lb.CV, ktail);
            if (LATE && o + 1 == NO && MODE < 2) la.template load_all<MODE == 1>(ktail);  // A of stage kt + 2
          }
        }
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
#pragma unroll
  for (int o = 0; o < NOA; ++o)
    if (la.koct == 0) ex[la.row0 + la.step(o)] = scale_exp(la.s[o]);
#pragma unroll
  for (int o = 0; o < NOB; ++o)
    if (lb.koct == 0) ex[BM + lb.row0 + lb.step(o)] = scale_exp(lb.s[o]);
  __syncthreads();
  int pc[TN];
  unsigned worst = 0;
  const unsigned odd = (unsigned)l16 << 31;
#pragma unroll
  for (int j = 0; j < TN; ++j) pc[j] = ex[BM + wn * WN + 16 * j + l16];
#pragma unroll
  for (int i = 0; i < TM; ++i)
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
  const int r0 = m0 + wm * WM, c0 = n0 + wn * WN;
  if (__any(worst >= 0x7f800000u)) fp32_tile<TM, TN, AK, BKC>(g, acc, r0, c0, kbeg, kend, g16, l16);
  write_tiles(g, acc, r0, c0, g16, l16, m0 + BM <= g.M && n0 + BN <= g.N);
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
