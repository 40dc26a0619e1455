// Scalar arithmetic shared by the NF4 kernels.  Everything here compiles for the host as well as for
// gfx950, so the rounding rules can be tested exhaustively on a CPU.
//
// The eager reference performs every step of to_nf4 / get_original_weight in the weight's own dtype
// (torchao NF4Tensor, called from torchtune/modules/peft/lora.py:86 and
// torchtune/modules/low_precision/nf4_linear.py:49).  For bfloat16 that means: compute in fp32, round to
// nearest-even bf16 after every single operation.  `Arith<BF16>::rnd` is that rounding step.
#pragma once
#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#define TT_HD __host__ __device__ __forceinline__
#else
#define TT_HD inline
#endif

namespace ttamd {

// The 16 NormalFloat4 code points (QLoRA paper, table in appendix E); each is exactly representable in fp32.
#define TT_NF4_TABLE                                                                                              \
  {-1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f, -0.28444138169288635f,              \
   -0.18477343022823334f, -0.09105003625154495f, 0.0f, 0.07958029955625534f, 0.16093020141124725f,               \
   0.24611230194568634f, 0.33791524171829224f, 0.44070982933044434f, 0.5626170039176941f, 0.7229568362236023f,  \
   1.0f}

TT_HD uint32_t f32_bits(float f) {
  uint32_t u;
#if defined(__HIP_DEVICE_COMPILE__)
  u = __builtin_bit_cast(uint32_t, f);
#else
  memcpy(&u, &f, 4);
#endif
  return u;
}
TT_HD float bits_f32(uint32_t u) {
  float f;
#if defined(__HIP_DEVICE_COMPILE__)
  f = __builtin_bit_cast(float, u);
#else
  memcpy(&f, &u, 4);
#endif
  return f;
}

// fp32 -> bf16 bit pattern, round to nearest even, NaN stays a (quiet) NaN.
TT_HD uint16_t f32_to_bf16_bits(float f) {
  uint32_t u = f32_bits(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x0040u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
TT_HD float bf16_bits_to_f32(uint16_t b) { return bits_f32(((uint32_t)b) << 16); }

// fp32 value rounded to bf16 precision, returned as fp32.
TT_HD float round_to_bf16(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (float)(__bf16)f;  // v_cvt_pk_bf16_f32: round to nearest even
#else
  return bf16_bits_to_f32(f32_to_bf16_bits(f));
#endif
}

template <bool BF16>
struct Arith {
  static TT_HD float rnd(float f) { return BF16 ? round_to_bf16(f) : f; }
};

// Index of the NF4 code nearest to `scaled` under the reference's rule: distances |scaled - nf4[j]| are
// computed and rounded in the tensor dtype, and the FIRST minimum wins (torch.argmin over dim=-1).
// `scaled` must already be rounded to the dtype.  NaN (0/0 from an all-zero block) yields index 0, the
// position torch.argmin reports for an all-NaN row.
template <bool BF16>
TT_HD int nf4_nearest_code(float scaled) {
  const float tab[16] = TT_NF4_TABLE;
  int best = 0;
  float bestd = __builtin_fabsf(Arith<BF16>::rnd(scaled - Arith<BF16>::rnd(tab[0])));
#pragma unroll
  for (int j = 1; j < 16; ++j) {
    float d = __builtin_fabsf(Arith<BF16>::rnd(scaled - Arith<BF16>::rnd(tab[j])));
    if (d < bestd) {  // strict: ties keep the lower index; NaN never wins
      bestd = d;
      best = j;
    }
  }
  return best;
}

// ---- code search by bins ---------------------------------------------------------------------------
// Along the scaled values -1 .. 1 the nearest code only grows, in steps of one, at 15 edges that lie at least 0.08 apart.
// 1/16-wide bins therefore hold one edge at most: an entry per bin says the code below its edge and the edge itself, so a
// code costs one table read and one comparison.  Bins are addressed by the low bits of 64 * t + 1.5 * 2^23: the byte
// offset of a 4-byte entry, 0x00 .. 0x40 for t >= 0 and 0xC0 .. 0xFC below.
constexpr int kNf4Bins = 64;
constexpr uint32_t kNf4NoEdge = 0x7f000000u;  // 1.7e38: no scaled value is above it

TT_HD uint32_t nf4_bin_offset(float t) { return f32_bits(__builtin_fmaf(t, 64.0f, 12582912.0f)) & 0xfcu; }

// bfloat16: `t` = x * y with y = 1 / absmax to one unit in the last place, `entry` = the edge with the code below it in
// its low four bits.  The reference's value is the quotient rounded to bf16, whose edges lie halfway between two bf16
// values (9-bit significands): a quotient of two 8-bit significands is such an edge or at least 2^-17 of it away.  The
// stored edge is 16 - 32 units (2^-20 .. 2^-18) off to the side that its tie rounds away from, so neither the code bits
// nor the error of t (2^-22) ever decide.
TT_HD uint32_t nf4_code_below(uint32_t entry) { return entry & 15u; }
TT_HD bool nf4_above_edge_bf16(float t, uint32_t entry) { return t > bits_f32(entry); }

// float: the quotient itself, correctly rounded, against the smallest float of the code above the edge.  With
// y = RN(1 / m) two corrections of x * y give RN(x / m) (the residuals are exact: no operand near the ends of the range).
TT_HD float nf4_shared_quotient(float x, float m, float y) {
  float q = x * y;
  q = __builtin_fmaf(__builtin_fmaf(-q, m, x), y, q);
  return __builtin_fmaf(__builtin_fmaf(-q, m, x), y, q);
}

// absmax bit patterns [low, high) for which the above holds; others take the division and the search of the 16 codes
template <bool BF16>
struct Nf4FastRange {
  static constexpr uint32_t low = BF16 ? 0x04000000u : 0x1f800000u;   // 2^-119, 2^-64
  static constexpr uint32_t high = BF16 ? 0x7e800000u : 0x5f800000u;  // 2^126 (1 / m is normal), 2^64
};

template <bool BF16>
struct Nf4BinTable {
  static constexpr int kWords = BF16 ? kNf4Bins : 2 * kNf4Bins;  // edges; float: codes behind them
  uint32_t words[kWords];
};

// Fills the table from nf4_nearest_code; false if one of the premises above does not hold.
template <bool BF16>
inline bool nf4_fill_bins(Nf4BinTable<BF16>& out) {
  const float tab[16] = TT_NF4_TABLE;
  bool ok = nf4_nearest_code<BF16>(bits_f32(0x7fc00000u)) == 0 && nf4_nearest_code<BF16>(-1.0f) == 0 &&
            nf4_nearest_code<BF16>(1.0f) == 15;
  constexpr int kShift = BF16 ? 16 : 0;  // neighbours in the dtype are 1 << kShift apart as float bits
  auto value = [](int64_t order) {       // the dtype's values in ascending order, 0 = +0
    return order >= 0 ? bits_f32((uint32_t)order << kShift) : bits_f32(0x80000000u | ((uint32_t)(-order) << kShift));
  };
  auto order_of = [](float v) {
    const int64_t mag = (int64_t)((f32_bits(v) & 0x7fffffffu) >> kShift);
    return v < 0 ? -mag : mag;
  };
  float first[16], edge[16];  // of code k: its smallest value, and the value from which t counts as k
  for (int k = 1; k < 16; ++k) {
    int64_t lo = order_of(Arith<BF16>::rnd(tab[k - 1])), hi = order_of(Arith<BF16>::rnd(tab[k]));
    while (hi - lo > 1) {
      const int64_t mid = lo + (hi - lo) / 2;
      (nf4_nearest_code<BF16>(value(mid)) >= k ? hi : lo) = mid;
    }
    ok = ok && nf4_nearest_code<BF16>(value(lo)) == k - 1 && nf4_nearest_code<BF16>(value(hi)) == k;
    first[k] = value(hi);
    edge[k] = BF16 ? 0.5f * (value(lo) + value(hi)) : value(hi);
    if (BF16) {
      const bool tie_up = (f32_bits(first[k]) >> 16 & 1u) == 0;  // ties go to the even neighbour
      const bool outwards = (edge[k] > 0) != tie_up;
      const uint32_t b = f32_bits(edge[k]);
      ok = ok && (b & 0x7fffu) == 0 && edge[k] != 0;
      edge[k] = bits_f32((outwards ? b + 16u : b - 32u) | (uint32_t)(k - 1));
    }
  }
  for (int b = 0; b < kNf4Bins; ++b) {
    const int j = b <= 16 ? b : b - kNf4Bins;
    uint32_t e = kNf4NoEdge, below = 0;
    for (int k = 1; k < 16; ++k) {
      const int at = (int)(nf4_bin_offset(edge[k]) >> 2);
      const int jk = at <= 16 ? at : at - kNf4Bins;
      // the value that picks the bin carries t's error: the edge's surroundings must lie in the same bin
      ok = ok && nf4_bin_offset(edge[k] * (1.0f + 0x1p-12f)) >> 2 == (uint32_t)at &&
           nf4_bin_offset(edge[k] * (1.0f - 0x1p-12f)) >> 2 == (uint32_t)at;
      if (jk < j) below = (uint32_t)k;
      if (jk == j) {
        ok = ok && e == kNf4NoEdge;
        e = f32_bits(edge[k]);
      }
    }
    out.words[b] = BF16 ? ((e & ~15u) | below) : e;
    if (!BF16) out.words[kNf4Bins + b] = below;
  }
  return ok;
}

// Dequantised value of one block scaler: (int8 / factor) rounded to dtype, plus mean, rounded again.
template <bool BF16>
TT_HD float nf4_block_scaler(int q, float factor, float mean) {
  float s = Arith<BF16>::rnd((float)q / factor);
  return Arith<BF16>::rnd(s + mean);
}

}  // namespace ttamd
