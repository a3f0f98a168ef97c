// bf16-MFMA GEMM over strided operands of any alignment, in fp32 and bf16
// (gfx950 v_mfma_f32_32x32x16_bf16, fp32 sums): the engine of the
// reference-layout fused_linear_transpose op in fp32, and in bf16 for the
// layouts the direct-to-LDS kernels do not take (a time axis that is not a
// multiple of their tile, operands that start off a 16-byte boundary).
//
//   C(m, n) = sum_{ko < KO} sum_{ki < kin} A(m, ko, ki) B(n, ko, ki)
//   A(m, ko, ki) at A + m sam + ko sako + ki saki (+ z sab for batch z), B alike
//
// fp32 operands are split exactly into three bf16 pieces, x = x1 + x2 + x3 (each
// the rest rounded to nearest: 8 + 8 + 8 bits of the significand; scaled, so that
// subnormal pieces lose no bits either: kSplitScale), and a
// product is six MFMA terms, smallest first: x3 y1, x1 y3, x2 y2, x2 y1, x1 y2,
// x1 y1.  The three left out come to at most 2^-24 of a product (x2 y3 and x3 y2
// 2^-25 each), 2^-27.5 in the mean.  The bf16 MFMA was seen to round correctly
// where the accumulator is the largest addend, and to cut addends below the last bit
// of the largest elsewhere.  So x1 y1 has an accumulator to itself, with K / 16
// roundings where the fp32 MFMA takes K / 2, and the five smaller terms (2^-8 of it)
// share another; they are added at the end.  Worst case, with every cut bit set,
// (K / 15 + 18) 2^-24 of the sum of the products' magnitudes, against K 2^-24 in
// fp32 arithmetic; reductions of up to 16 indices, which show the cut bits, run on
// the fp32 MFMA (split_blocks_f32).
// A bf16 MFMA term is 16 times as fast as the fp32 MFMA (2.5 against 0.157
// PFLOP/s nominal), six of them 2.7 times.  Non-finite results send the
// wavefront's part of the tile through the fp32 MFMA too (an infinity has
// no such split, nor has a value that the scale takes past the largest bf16), so
// infinities and NaNs come out as fp32 arithmetic gives them; a tile that meets
// one in its first step goes there at once.  (B = 8, T = 1024, K = 768, F = 2322,
// all NaN: forward 393, both gradients 884 us, against 265 and 617 for the fp32
// MFMA kernel; one NaN 289 and 484.)
// bf16 operands are one piece: the products are exact, as they always were.
//
// Measured on MI355X against the fp32-MFMA kernel before it (128 x 128 tiles,
// quads, one element per load off a 16-byte boundary), 2-norm errors against
// float64, normally distributed operands:
//   fp32 B = 32, T = 1024, K = 768, F = 2322: errors 5.0e-7 -> 1.6e-7 (forward),
//     8.6e-7 -> 2.9e-7 (grad_x), 9.0e-7 -> 3.1e-7 (grad_weight); with all six terms in
//     one accumulator 4.2e-7, 7.5e-7, 9.1e-7 (B = 8 of it 177 and 383 us);
//   fp32 B = 8: 265 -> 185 and 617 -> 388 us; B = 2, T = 16: 57.6 -> 16, 179 -> 60;
//     M = 300 with K = 1 / 16: 2.5e-8 and 7.5e-8 as before;
//   bf16 B = 20, T = 1501, K = 768, F = 2322: 971 -> 194 us (551 TFLOP/s), 3265
//     -> 408 us (524); B = 5, T = 1501, K = 512, F = 1040: 117 -> 25, 328 -> 75.
// What bounds the fp32 form: the matrix cores, busy half of the cycles (32 per MFMA,
// counted) at the clock that random operands leave, and the conversion beside them;
// halving its instructions gained 3%.
//
// 128 x 128 output tiles, 4 wavefronts of 64 x 64, three workgroups per CU in bf16
// and two in fp32 (so that one wavefront's barrier, load wait or conversion leaves
// the matrix core to the SIMD's others; fp32's second accumulator takes the
// registers of a third: with one accumulator, each step's terms summed from zero and
// added to it, three fit, but the additions cost more: 197 and 443 us against 190
// and 404); 64 x 64 tiles where those are too few.
// The global loads run two steps ahead in registers, and the next step is
// converted into the other of two LDS stages while this one runs its MFMAs; one
// barrier per step.
//
// An operand must be contiguous along its reduction (kSplitKC) or its rows
// (kSplitRC).  A thread loads chunks of 8 consecutive elements -- aligned
// to an element only: an odd bf16 chunk is read as whole dwords and shifted --
// and writes them to LDS as 16-byte chunks in the operand's own orientation:
//   KC  [row][k]: chunk c of row r at slot c ^ ((r / phase) & (chunks - 1)), phase
//       the rows of a 256-byte bank window, read with ds_read_b128;
//   RC  [k][row]: row-chunk c of k-row k at slot c ^ (4 (k & 3)), read with
//       ds_read_b64_tr_b16;
// both fragment reads are then free of bank conflicts.
//
// Whole steps never straddle an outer index: each ko has kin / BK of them, and where
// kin is not a multiple, its last indices go into steps of their own, packed over
// the outer indices (read element by element).  A step for each ko's would be up to
// 16 times the work: grad_weight of many short sequences, B = 64, T = 5, K = 128, F =
// 390 in fp32, both gradients 147 -> 60 us, bf16 76 -> 39.  A workgroup runs its
// whole steps first, pipelined, then the packed ones.  Split-K: blockIdx.z = batch *
// splits + split; split s takes the whole steps [s split_whole, (s + 1) split_whole)
// and the last indices of the outer indices [s split_tail, (s + 1) split_tail), and
// sums them into C + s scs.
#pragma once

#include "ltv_gemm_dma.hpp"

#include <cfloat>

namespace ltv {

enum SplitLayout { kSplitKC = 0, kSplitRC = 1 };

constexpr int kSplitThreads = 256;  // 4 wavefronts, 2 x 2

// fp32 operands are split at 2^24 times their value: the last bit of the
// smallest subnormal then lies at 2^-125, so every piece of every operand is a
// normal bf16 number or zero and the split is exact.  Sums are scaled back once,
// when they are stored.  (Operands from 2^104 and sums from 2^80 on overflow so
// and take the non-finite path.)
constexpr float kSplitScale = 16777216.0f;
constexpr float kSplitUnscale = 1.0f / (kSplitScale * kSplitScale);

// Pieces per element, and the k-step of a tile of R = 128 or 64 rows.
template <typename TI>
struct SplitTraits {
  static constexpr int kPieces = sizeof(TI) == 4 ? 3 : 1;
  static constexpr int kWgPerCu = sizeof(TI) == 4 ? 2 : 3;  // of 128 x 128 tiles
  __host__ __device__ static constexpr int bk(int R) { return sizeof(TI) == 4 && R == 128 ? 16 : 32; }
};

struct SplitArgs {
  const void* A;
  int64_t sam, sako, saki, sab;
  const void* B;
  int64_t sbn, sbko, sbki, sbb;
  void* C;
  int64_t scm, scn, scb, scs;  // output strides: row, column, batch, split
  int M, N, KO, kin;
  int split_whole;  // whole k-steps (of the KO (kin / BK)) per split
  int split_tail;   // outer indices whose last, partial range a split takes
  int splits;
};

// One operand of one workgroup: its rows [row0, row0 + 128).
template <typename TI>
struct SplitOperand {
  const TI* p;  // at the workgroup's batch
  int64_t sr, sko, ski;
  int rows, kin, row0;
  bool odd;  // bf16: some chunk may start inside a dword
};

typedef uint32_t u32x4a4_t __attribute__((ext_vector_type(4), aligned(4)));

// A thread's chunks of one operand tile, as loaded.
template <typename TI, int R>
struct SplitRaw {
  static constexpr int BK = SplitTraits<TI>::bk(R);
  static constexpr int NC = R * BK / 8 / kSplitThreads;  // chunks per thread
  static constexpr int W = sizeof(TI) == 4 ? 8 : 5;  // dwords (bf16: one more, for odd starts)
  static_assert(NC >= 1 && NC * 8 * kSplitThreads == R * BK, "whole chunks per thread");
  uint32_t w[NC][W];

  // fp32: whether an element leaves the range in which it is split (or is none)
  __device__ __forceinline__ int past_range() const {
    bool past = false;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        past = past || !(fabsf(__uint_as_float(w[c][i])) < FLT_MAX / kSplitScale);
    return past;
  }
};

// Where a step that is read element by element starts (load_checked).
struct SplitStep {
  int ko, k0, r, per;
};

// Global -> registers -> LDS staging of one R-row x BK tile.
template <typename TI, int L, int R>
struct SplitStager {
  using Raw = SplitRaw<TI, R>;
  static constexpr int E = sizeof(TI);
  static constexpr int BK = Raw::BK, NP = SplitTraits<TI>::kPieces, NC = Raw::NC;
  static constexpr int CPR = BK / 8;           // chunks per KC row
  static constexpr int kPlane = R * BK * 2;    // bytes of one piece's plane

  // chunk c at ko = 0, k0 = 0.  Rows past the operand: row 0.  An RC chunk that
  // the operand's end cuts is read `early` rows early, to end with it, and
  // shifted into place when it is stored; with fewer rows than a chunk it is read
  // on into the next k's rows, whose results are not stored.
  const TI* rp[NC];
  uint32_t early;

  // row (KC) or first row (RC), and k within the step, of chunk c
  __device__ __forceinline__ static int row_of(int c) {
    const int q = threadIdx.x + kSplitThreads * c;
    return L == kSplitKC ? q / CPR : 8 * (q % (R / 8));
  }
  __device__ __forceinline__ static int k_of(int c) {
    const int q = threadIdx.x + kSplitThreads * c;
    return L == kSplitKC ? 8 * (q % CPR) : q / (R / 8);
  }

  __device__ __forceinline__ void setup(const SplitOperand<TI>& op) {
    // (an RC thread's chunks share their rows)
    const int over = op.row0 + row_of(0) + 8 - op.rows;
    early = L == kSplitRC && over > 0 && over < 8 && op.rows >= 8 ? (uint32_t)over : 0u;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int row = op.row0 + row_of(c);
      const int64_t r = row < op.rows ? row - (int)early : 0;
      rp[c] = L == kSplitKC ? op.p + r * op.sr + k_of(c) : op.p + r + (int64_t)k_of(c) * op.ski;
    }
  }

  // 8 elements from p (aligned to an element)
  __device__ __forceinline__ static void load_chunk(Raw& o, int c, const TI* p, bool odd) {
    if constexpr (E == 4) {
      const u32x4a4_t a = *reinterpret_cast<const u32x4a4_t*>(p);
      const u32x4a4_t b = *reinterpret_cast<const u32x4a4_t*>(p + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        o.w[c][i] = a[i];
        o.w[c][4 + i] = b[i];
      }
    } else {
      const uintptr_t a = reinterpret_cast<uintptr_t>(p);
      const uint32_t* q = reinterpret_cast<const uint32_t*>(a & ~(uintptr_t)3);
      const u32x4a4_t v = *reinterpret_cast<const u32x4a4_t*>(q);
#pragma unroll
      for (int i = 0; i < 4; ++i) o.w[c][i] = v[i];
      if (odd) {
        // an odd chunk ends in the next dword; an even one reads no further
        o.w[c][4] = q[(a & 2u) != 0 ? 4 : 0];
      }
    }
  }

  // A step inside the reduction: off elements from the first one.
  __device__ __forceinline__ void load(Raw& o, const SplitOperand<TI>& op, int64_t off) const {
#pragma unroll
    for (int c = 0; c < NC; ++c) load_chunk(o, c, rp[c] + off, op.odd);
  }

  // Any step, element by element, to chunks that start on a dword: its first n
  // indices are (at.ko, at.k0 + at.r), ..., at.per of them (from at.k0 on) to an
  // outer index.
  __device__ __forceinline__ void load_checked(Raw& o, const SplitOperand<TI>& op,
                                               const SplitStep& at, int n) const {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int row = op.row0 + row_of(c), k = k_of(c);
      int ko = at.ko + (at.r + k) / at.per, r = (at.r + k) % at.per;
      const TI* p = rp[c] + early - (int64_t)k * op.ski;  // at ko = 0, k = 0
      const TI* q = p + (ko * op.sko + (at.k0 + r) * op.ski);
      // valid elements of the chunk, from its first on
      int m = L == kSplitKC ? (row < op.rows ? n - k : 0) : (k < n ? op.rows - row : 0);
      m = m < 0 ? 0 : m > 8 ? 8 : m;
#pragma unroll
      for (int i = 0; i < Raw::W; ++i) o.w[c][i] = 0u;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < m) {
          if constexpr (E == 4)
            o.w[c][e] = __float_as_uint(*q);
          else
            o.w[c][e >> 1] |= (uint32_t)*q << (16 * (e & 1));
          ++q;
          if (L == kSplitKC && ++r == at.per) {
            r = 0;
            ++ko;
            q = p + (ko * op.sko + at.k0 * op.ski);
          }
        }
    }
  }

  // The chunks as bf16 pieces to the planes at lds.  CHECKED: from
  // load_checked; else from load at the same `off`.
  template <bool CHECKED>
  __device__ __forceinline__ void store(Raw& o, char* lds, const SplitOperand<TI>& op,
                                        int64_t off) const {
    const bool cut = !CHECKED && L == kSplitRC && op.row0 + R > op.rows && op.rows % 8 != 0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int r = row_of(c), k = k_of(c);
      // (rows past the operand hold row 0 or zeros: their results are not stored)
      uint32_t at;
      if (L == kSplitKC) {
        constexpr int kRow = BK * 2, kPhase = 256 / kRow;
        at = (uint32_t)(r * kRow + (((k >> 3) ^ ((r / kPhase) & (CPR - 1))) << 4));
      } else {
        at = (uint32_t)(k * (R * 2) + (((r >> 3) ^ rc_swizzle(k)) << 4));
      }
      uint4* d = reinterpret_cast<uint4*>(lds + at);
      if constexpr (E == 2) {
        if (!CHECKED && op.odd) {
          const uint32_t sh = (uint32_t)(reinterpret_cast<uintptr_t>(rp[c] + off) & 2u) << 3;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o.w[c][i] = __builtin_amdgcn_alignbit(o.w[c][i + 1], o.w[c][i], sh);
        }
        if (cut) shift_down<4, 2>(o.w[c], early);
        d[0] = make_uint4(o.w[c][0], o.w[c][1], o.w[c][2], o.w[c][3]);
      } else {
        if (cut) shift_down<8, 1>(o.w[c], early);
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = __uint_as_float(o.w[c][e]) * kSplitScale;
        static_for<NP>([&](auto pc) {
          constexpr int p = decltype(pc)::value;
          uint32_t q[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            q[i] = cvt_pk_bf16(x[2 * i], x[2 * i + 1]);
            if (p + 1 < NP) {
              // the rest, exact: x - (1, 0) . q and x - (0, 1) . q
              x[2 * i] = rest(q[i], 0x0000bf80u, x[2 * i]);
              x[2 * i + 1] = rest(q[i], 0xbf800000u, x[2 * i + 1]);
            }
          }
          d[p * (kPlane / 16)] = make_uint4(q[0], q[1], q[2], q[3]);
        });
      }
    }
  }

  // x + q . m for a pair of bf16 q and m = (-1, 0) or (0, -1): one instruction
  // (v_dot2_f32_bf16) where widening q and subtracting takes two.  m goes through
  // a register: the pair (-1, 0) written as the instruction's inline -1.0 measured
  // as (0, -1).
  __device__ __forceinline__ static float rest(uint32_t q, uint32_t m, float x) {
    asm("" : "+s"(m));
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, q),
                                           __builtin_bit_cast(bf16x2_t, m), x, false);
  }

  // The first N dwords of w (EPD elements each) moved down by n < 8 elements,
  // zeros following.
  template <int N, int EPD>
  __device__ __forceinline__ static void shift_down(uint32_t (&w)[Raw::W], uint32_t n) {
    if (EPD == 2) {
      const uint32_t sh = 16u * (n & 1u);
#pragma unroll
      for (int i = 0; i < N; ++i)
        w[i] = __builtin_amdgcn_alignbit(i + 1 < N ? w[i + 1] : 0u, w[i], sh);
    }
    const uint32_t m = n / EPD;
    static_for<3>([&](auto lc) {
      constexpr int step = 1 << decltype(lc)::value;
      if constexpr (step < N) {
        const bool on = (m & step) != 0;
#pragma unroll
        for (int i = 0; i < N; ++i) w[i] = on ? (i + step < N ? w[i + step] : 0u) : w[i];
      }
    });
  }

  // Slot swizzle of k-row k of an RC tile: the four k-rows one 16-lane group of
  // ds_read_b64_tr_b16 reads land in four disjoint 64-byte windows (rows of
  // 256 bytes, or two to the 256-byte bank window).
  __device__ __forceinline__ static int rc_swizzle(int k) {
    return R == 128 ? 4 * (k & 3) : 4 * ((k >> 1) & 1);
  }

  // MFMA operand fragment (8 consecutive k of row rb + lane % 32) of k16 sub-step t.
  __device__ __forceinline__ static bf16x8_t frag(const char* plane, int rb, int t, int lane) {
    typedef __attribute__((address_space(3))) const char lds_char;
    lds_char* base = (lds_char*)plane;
    if (L == kSplitRC) {
      const int g = lane >> 4, s = lane & 15;
      const int row = rb + (g & 1) * 16 + 4 * (s & 3);
      const int k = t * 16 + (g >> 1) * 8 + (s >> 2);
      typedef __attribute__((address_space(3))) i16x4_t lds_i16x4;
      lds_char* p0 = base + k * (R * 2) + (((row >> 3) ^ rc_swizzle(k)) << 4) + (row & 7) * 2;
      lds_char* p1 = p0 + 4 * (R * 2);  // k + 4: the same swizzle
      const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)p0);
      const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)p1);
      typedef short i16x8_t __attribute__((ext_vector_type(8)));
      const i16x8_t v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      return __builtin_bit_cast(bf16x8_t, v);
    }
    constexpr int kRow = BK * 2, kPhase = 256 / kRow;
    const int r = rb + (lane & 31), c = 2 * t + (lane >> 5);
    return __builtin_bit_cast(
        bf16x8_t, *(__attribute__((address_space(3))) const u32x4_t*)(
                      base + r * kRow + ((c ^ ((r / kPhase) & (CPR - 1))) << 4)));
  }
};

// WB neighbouring blocks of 32 x 32 (A rows m0.., B rows n0..) over the whole
// steps [w0, w1) and the ends of the outer indices [t0, t1), on the fp32
// MFMA straight from memory: where a result is not finite, and for reductions too
// short to split.  Which four of eight consecutive k a lane holds is free, as long
// as it is the same in A and B: each half of the wavefront reads four consecutive
// ones (KC: one 16-byte load), eight k ahead of the MFMAs.  Rows past the operand
// read its last one (unused).
template <int L>
__device__ __forceinline__ void split_f32_load(const SplitOperand<float>& op, const float* p,
                                               float (&o)[4]) {
  if constexpr (L == kSplitKC) {
    const u32x4a4_t v = *reinterpret_cast<const u32x4a4_t*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __uint_as_float(v[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = p[i * op.ski];
  }
}

template <int LA, int LB, int WB, int BK>
__device__ __forceinline__ void split_blocks_f32(const SplitOperand<float>& oa,
                                                 const SplitOperand<float>& ob, int m0, int n0,
                                                 int w0, int w1, int t0, int t1, int wpb,
                                                 int lane, f32x16_t (&acc)[WB]) {
  const int h = lane >> 5;
  const float* pa = oa.p + (int64_t)min(m0 + (lane & 31), oa.rows - 1) * oa.sr;
  const float* pb[WB];
#pragma unroll
  for (int b = 0; b < WB; ++b) {
    pb[b] = ob.p + (int64_t)min(n0 + 32 * b + (lane & 31), ob.rows - 1) * ob.sr;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[b][v] = 0.0f;
  }
  auto mfma = [&](int b, float x, float y) {
    acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc[b], 0, 0, 0);
  };
  if (w1 > w0) {
    int ko = w0 / wpb, k = (w0 - ko * wpb) * BK;
    float x[2][4], y[2][WB][4];
    auto load = [&](auto setc) {
      constexpr int set = decltype(setc)::value;
      const int64_t fa = ko * oa.sko + (k + 4 * h) * oa.ski;
      const int64_t fb = ko * ob.sko + (k + 4 * h) * ob.ski;
      split_f32_load<LA>(oa, pa + fa, x[set]);
#pragma unroll
      for (int b = 0; b < WB; ++b) split_f32_load<LB>(ob, pb[b] + fb, y[set][b]);
    };
    auto mfmas = [&](auto setc) {
      constexpr int set = decltype(setc)::value;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int b = 0; b < WB; ++b) mfma(b, x[set][i], y[set][b][i]);
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    const int groups = (w1 - w0) * (BK / 8);  // of 8 k: an even number
    auto next = [&](int g) {
      if (g + 1 < groups) {  // (else the last group again, unused)
        k += 8;
        if (k == wpb * BK) {
          k = 0;
          ++ko;
        }
      }
    };
    load(S0{});
    for (int g = 0; g < groups; g += 2) {
      next(g);
      load(S1{});
      mfmas(S0{});
      next(g + 1);
      load(S0{});
      mfmas(S1{});
    }
  }
  for (int ko = t0; ko < t1; ++ko)
    for (int kk = wpb * BK; kk < oa.kin; kk += 2) {
      const int k = kk + h;
      const float x = k < oa.kin ? pa[ko * oa.sko + k * oa.ski] : 0.0f;
#pragma unroll
      for (int b = 0; b < WB; ++b)
        mfma(b, x, k < oa.kin ? pb[b][ko * ob.sko + k * ob.ski] : 0.0f);
    }
}

// WB x WB blocks of 32 x 32 per wavefront: tiles of R = 64 WB rows of A and of B.
template <typename TI, typename TO, int LA, int LB, int WB>
__global__ void __launch_bounds__(kSplitThreads, WB == 2 ? SplitTraits<TI>::kWgPerCu : 3)
gemm_split_kernel(const SplitArgs g) {
  constexpr int R = 64 * WB;
  using StA = SplitStager<TI, LA, R>;
  using StB = SplitStager<TI, LB, R>;
  constexpr int BK = StA::BK, NP = StA::NP, kPlane = StA::kPlane;
  __shared__ __attribute__((aligned(1024))) char lds_a[2][NP * kPlane];
  __shared__ __attribute__((aligned(1024))) char lds_b[2][NP * kPlane];

  // workgroup w (dispatch order) runs on XCD w % 8: deal the tiles to the XCDs
  // in contiguous ranges (n-tiles fastest), so tiles sharing an operand tile
  // share that XCD's L2.  XCD x holds the workgroups x, x + 8, ... < total:
  // q + (x < r) of them (q, r = total / 8, total % 8), tiles from x q + min(x, r).
  const int gx = gridDim.x, gy = gridDim.y;
  const int64_t total = (int64_t)gx * gy * gridDim.z;
  const int64_t wg = blockIdx.x + (int64_t)gx * (blockIdx.y + (int64_t)gy * blockIdx.z);
  const int64_t xcd = wg % 8, q = total / 8, r = total % 8;
  const int64_t u = xcd * q + (xcd < r ? xcd : r) + wg / 8;
  const int tx = (int)(u % gx), ty = (int)((u / gx) % gy), z = (int)(u / ((int64_t)gx * gy));
  const int batch = z / g.splits, split = z - batch * g.splits;
  const int m0 = ty * R, n0 = tx * R;

  auto odd = [](const void* p, int64_t a, int64_t b, int64_t c) {
    return sizeof(TI) == 2 && (((reinterpret_cast<uintptr_t>(p) >> 1) | a | b | c) & 1) != 0;
  };
  const SplitOperand<TI> oa{reinterpret_cast<const TI*>(g.A) + (int64_t)batch * g.sab, g.sam,
                            g.sako, g.saki, g.M, g.kin, m0,
                            odd(g.A, g.sab, g.sako, LA == kSplitKC ? g.sam : g.saki | g.M)};
  const SplitOperand<TI> ob{reinterpret_cast<const TI*>(g.B) + (int64_t)batch * g.sbb, g.sbn,
                            g.sbko, g.sbki, g.N, g.kin, n0,
                            odd(g.B, g.sbb, g.sbko, LB == kSplitKC ? g.sbn : g.sbki | g.N)};

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = (wave & 1) * (32 * WB), wn = (wave >> 1) * (32 * WB);

  f32x16_t acc[WB][WB];
#pragma unroll
  for (int a = 0; a < WB; ++a)
#pragma unroll
    for (int b = 0; b < WB; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;
  // fp32: the sums of the terms below x1 y1
  f32x16_t low[NP == 3 ? WB : 1][NP == 3 ? WB : 1];
  if constexpr (NP == 3) {
#pragma unroll
    for (int a = 0; a < WB; ++a)
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) low[a][b][v] = 0.0f;
  }

  StA sa;
  StB sb;
  sa.setup(oa);
  sb.setup(ob);
  auto mfmas = [&](int cur) {
#pragma unroll
    for (int t = 0; t < BK / 16; ++t) {
      bf16x8_t fb[NP][WB];
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int b = 0; b < WB; ++b)
          fb[p][b] = StB::frag(lds_b[cur] + p * kPlane, wn + 32 * b, t, lane);
#pragma unroll
      for (int a = 0; a < WB; ++a) {
        bf16x8_t fa[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p)
          fa[p] = StA::frag(lds_a[cur] + p * kPlane, wm + 32 * a, t, lane);
#pragma unroll
        for (int b = 0; b < WB; ++b) {
          if constexpr (NP == 3) {
            // smallest terms first; x1 y1 by itself
            constexpr int kTerms[5][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}};
            static_for<5>([&](auto tc) {
              constexpr int pa = kTerms[decltype(tc)::value][0];
              constexpr int pb = kTerms[decltype(tc)::value][1];
              low[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[pa], fb[pb][b], low[a][b],
                                                                  0, 0, 0);
            });
          }
          acc[a][b] =
              __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[0], fb[0][b], acc[a][b], 0, 0, 0);
        }
      }
    }
  };
  SplitRaw<TI, R> ra[2], rb[2];

  // The whole steps, an even number of them, pipelined: while step s runs, step
  // s + 1 (loaded a step earlier) is converted and written to the other stage
  // and step s + 2 is loaded, so a load has two steps to arrive.  Past the end
  // the last step is loaded and stored again, unused: no branch in the loop.
  const int wpb = g.kin / BK;  // whole steps per outer index
  const int w0 = split * g.split_whole, w1 = min(g.KO * wpb, w0 + g.split_whole);
  // (an RC operand with fewer rows than a chunk is read past its row: every step but
  // the reduction's last whole one has at least BK more k behind it)
  const bool few = (LA == kSplitRC && g.M < 8) || (LB == kSplitRC && g.N < 8);
  const int ahead = w1 - w0 - (few && w1 == g.KO * wpb ? 1 : 0);
  const int np = ahead > 0 ? ahead & ~1 : 0;
  // fp32: the whole tile on the fp32 MFMA, for reductions of up to 16 indices.
  // (K = 1 on the bf16 MFMA: up to 1.5e-7 of the product, against 6e-8 rounded
  // once; K = 2 3.4e-8 of the result in 2-norm against 3.1e-8; K = 4 3.2e-8 against
  // 4.0e-8, but 7.6e-8 against 8e-9 for K = 7 equal products)
  bool direct = NP == 3 && (int64_t)g.KO * g.kin <= 16;
  if (np > 0 && !direct) {
    int ko = w0 / wpb, ki = w0 - ko * wpb, left = np;
    int64_t offa[2], offb[2];
    auto load = [&](auto setc) {
      constexpr int set = decltype(setc)::value;
      offa[set] = (int64_t)ko * oa.sko + (int64_t)(ki * BK) * oa.ski;
      offb[set] = (int64_t)ko * ob.sko + (int64_t)(ki * BK) * ob.ski;
      sa.load(ra[set], oa, offa[set]);
      sb.load(rb[set], ob, offb[set]);
      const int nki = ki + 1 < wpb ? ki + 1 : 0, nko = ki + 1 < wpb ? ko : ko + 1;
      --left;
      ki = left > 0 ? nki : ki;
      ko = left > 0 ? nko : ko;
    };
    auto store = [&](auto setc) {
      constexpr int set = decltype(setc)::value;
      sa.template store<false>(ra[set], lds_a[set], oa, offa[set]);
      sb.template store<false>(rb[set], lds_b[set], ob, offb[set]);
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    load(S0{});
    load(S1{});
    // an operand past the scaled range in the first step: the results will not be
    // finite, and the tile need not be run twice
    if constexpr (NP == 3) direct = __syncthreads_or(ra[0].past_range() | rb[0].past_range());
    store(S0{});
    __syncthreads();
    for (int s = 0; s < (direct ? 0 : np); s += 2) {
      // (a stage is refilled after the barrier that ended its last reads)
      load(S0{});
      mfmas(0);
      store(S1{});
      __syncthreads();
      load(S1{});
      mfmas(1);
      store(S0{});
      __syncthreads();
    }
  }
  const int tail = g.kin - wpb * BK, tails = tail > 0 ? g.KO : 0;
  const int t0 = split * g.split_tail, t1 = min(tails, t0 + g.split_tail);
  // The steps left: the last whole ones, then the ends of the outer indices' ranges,
  // packed.
  if (!direct) {
    int tko = t0, tr = 0;
    int64_t left = (int64_t)(t1 - t0) * tail;
    for (int w = w0 + np; w < w1 || left > 0;) {
      const bool whole = w < w1;
      const int ko = whole ? w / wpb : tko;
      const SplitStep at{ko, whole ? (w - ko * wpb) * BK : wpb * BK, whole ? 0 : tr,
                         whole ? BK : tail};
      const int n = whole || left > BK ? BK : (int)left;
      sa.load_checked(ra[0], oa, at, n);
      sb.load_checked(rb[0], ob, at, n);
      sa.template store<true>(ra[0], lds_a[0], oa, 0);
      sb.template store<true>(rb[0], lds_b[0], ob, 0);
      __syncthreads();
      mfmas(0);
      __syncthreads();
      if (whole) {
        ++w;
      } else {
        left -= BK;
        tko += (tr + BK) / tail;
        tr = (tr + BK) % tail;
      }
    }
  }

  TO* C = reinterpret_cast<TO*>(g.C) + (int64_t)batch * g.scb + (int64_t)split * g.scs;
  // lane l of a block at (mb, nb) holds column nb + l % 32 and rows
  // mb + 8 (v / 4) + 4 (l / 32) + v % 4
  auto store_block = [&](int mb, int nb, const f32x16_t& c) {
    const int n = nb + (lane & 31);
    if (n >= g.N) return;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = mb + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if (m < g.M) io_traits<TO>::store(C + (int64_t)m * g.scm + (int64_t)n * g.scn, c[v]);
    }
  };
  if constexpr (NP == 3) {
#pragma unroll
    for (int a = 0; a < WB; ++a)
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[a][b][v] = (acc[a][b][v] + low[a][b][v]) * kSplitUnscale;
    bool bad = direct;
#pragma unroll
    for (int a = 0; a < WB; ++a)
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) bad = bad || !(fabsf(acc[a][b][v]) < INFINITY);
    if (__builtin_amdgcn_readfirstlane(__any(bad))) {
#pragma unroll 1
      for (int a = 0; a < WB; ++a) {
        f32x16_t c[WB];
        split_blocks_f32<LA, LB, WB, BK>(oa, ob, m0 + wm + 32 * a, n0 + wn, w0, w1, t0, t1, wpb,
                                         lane, c);
#pragma unroll
        for (int b = 0; b < WB; ++b) store_block(m0 + wm + 32 * a, n0 + wn + 32 * b, c[b]);
      }
      return;
    }
  }
#pragma unroll
  for (int a = 0; a < WB; ++a)
#pragma unroll
    for (int b = 0; b < WB; ++b)
      store_block(m0 + wm + 32 * a, n0 + wn + 32 * b, acc[a][b]);
}

}  // namespace ltv
