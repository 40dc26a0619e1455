// y = x . dequant(Wq)^T (+ bias) for the converted integer linears and up to a few hundred tokens: the 8da4w layer (int4
// values held in int8, per-group scale and zero point) and the weight-only 4w layer (two uint4 codes per byte, bf16 scale
// and floating-point zero point).  What Int8DynActInt4WeightLinear / WeightOnlyInt4Linear.forward otherwise do in two
// passes - write the dense bf16 weight, read it back in a library GEMM - streams the integer weight once: 1 or 0.5
// bytes per element instead of 5 or 4.5.
//
// The expanded values are the bits of ttamd_dequantize_per_group_int4 / _uint4, the products are summed in fp32 and the
// result is rounded to bf16 once: the arithmetic of the two-pass form up to the order of the fp32 sums.
//
// Two kernels, by the number of tokens:
//  * int4_stream_kernel (at most 16): bound by the weight stream.  A workgroup owns 16 or 32 weight rows and the whole
//    contraction; its waves take 128-wide chunks of K in turn, one in flight each while the one before it is multiplied.
//    Neighbouring waves then read neighbouring pieces of the rows.  The lane that feeds an MFMA holds 32 consecutive k of one
//    row; a chunk's codes, scales and x come by direct-to-LDS loads in row order and are read from there.  Partial sums
//    meet in LDS in wave order.
//  * int4_tile_kernel (more): the few-token kernel would read all of x in every workgroup (at 75 tokens nine times the
//    bytes of its weight rows).  Eight waves share 64 weight rows and up to 128 tokens; a weight fragment is expanded once per 128
//    tokens.  Launches of few tiles cut the contraction into slices (fp32 slabs, added in slice order by int4_reduce_kernel).
//
// Measured against dequantise + library GEMM (us, weights from HBM, launch gaps included; int8 / uint4):
//   14336 x 4096:  1 token 60 / 60 -> 17.7 / 15.0, 16 tokens 59 / 60 -> 25 / 16.7, 75 tokens 63 / 65 -> 31 / 26, 256 tokens 83 / 82 -> 59 / 54
//   4096 x 14336:  1 token 58 / 58 -> 16.5 / 13.5, 75 tokens 79 / 78 -> 33 / 26, 256 tokens 93 / 92 -> 61 / 49
//   1024 x 4096:   1 token 20 / 20 -> 6.1 / 5.1, 256 tokens 21 / 21 -> 16 / 14
// (at most 16 tokens with loads straight into the MFMA lanes and one wave's sum at the end: 26.4 / 19.0, 21.9 / 19.5 and 9.0 / 7.3 at
// one token; a read of the same bytes takes 14 / 6.5).
#include "common.h"
#include "fq_math.h"
#include "nf4_math.h"

#include <algorithm>
#include <type_traits>

#define TT_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

namespace ttamd {
namespace {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_pair(float lo, float hi) {
  bf16x2_t v;
  v.x = (__bf16)lo;
  v.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float lo_of(uint32_t d) { return bits_f32(d << 16); }
__device__ __forceinline__ float hi_of(uint32_t d) { return bits_f32(d & 0xffff0000u); }

// The eight uint4 codes of a dword (the even element in a byte's high nibble) as an MFMA operand: bf16(bf16((q - 8) * scale) + zero).
// A nibble under the exponent of 1024 is the half 1024 + q (1024 + 16 q), two to a dword; q - 8 is exact from there on and
// (q - 8) * scale is rounded to bf16 directly, whatever the scale (8 * scale overflows above 2^125).  A value rounded into the
// upper half of a dword is its own fp32.  37 instructions, spelled out: the compiler makes 60 - 75 of the plain expressions (one
// token of 14336 x 4096 18.1 us, 15.0 with these).
__device__ __forceinline__ u32x4_t uint4_operand(uint32_t codes, float sc, float z) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float sc16 = sc * 0.0625f;
  uint32_t half[4];  // [0], [1]: bytes 0 and 2, [2], [3]: bytes 1 and 3; 16 (q - 8) of the even and q - 8 of the odd elements
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const uint32_t c = codes >> (8 * b);
    uint32_t even, odd;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(even) : "v"(c), "s"(0x00f000f0u), "v"(0x64006400u));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(odd) : "v"(c), "s"(0x000f000fu), "v"(0x64006400u));
    asm("v_pk_add_f16 %0, %1, %2" : "=v"(half[2 * b]) : "v"(even), "s"(0xe480e480u));     // - 1152
    asm("v_pk_add_f16 %0, %1, %2" : "=v"(half[2 * b + 1]) : "v"(odd), "s"(0xe408e408u));  // - 1032
  }
  u32x4_t w;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const uint32_t even = half[2 * (b & 1)], odd = half[2 * (b & 1) + 1];
    float p0, p1, r0, r1;
    if (b < 2) {
      asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(p0) : "v"(even), "v"(sc16));
      asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(p1) : "v"(odd), "v"(sc));
    } else {
      asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(p0) : "v"(even), "v"(sc16));
      asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(p1) : "v"(odd), "v"(sc));
    }
    asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(r0) : "v"(p0));
    asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(r1) : "v"(p1));
    w[b] = pack_pair(r0 + z, r1 + z);
  }
  return w;
#else
  return u32x4_t{};
#endif
}

// Eight int8 values of two dwords: bf16((q - zero) * scale)
__device__ __forceinline__ u32x4_t int8_operand(uint32_t low, uint32_t high, float sc, float z) {
  u32x4_t w;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const uint32_t two = (d < 2 ? low : high) >> (16 * (d & 1));
    w[d] = pack_pair(((float)(int8_t)(two & 0xffu) - z) * sc, ((float)(int8_t)((two >> 8) & 0xffu) - z) * sc);
  }
  return w;
}

struct Int4Args {
  const uint16_t* x;     // [M, K] bf16
  const uint8_t* q;      // int8 [N, K] or packed uint4 [N, K/2]
  const void* scale;     // int8 form: [N, K/g]; uint4 form: bf16 [K/g, N, 2] (scale, zero)
  const void* zero;      // int8 form: [N, K/g] or null (= 0)
  const uint16_t* bias;  // [N] bf16 or null
  uint16_t* y;           // [M, N] bf16
  float* part;           // [slices, M, N] when the contraction is cut
  int M, N, K;
  int log2_group;        // >= 5
  int chunks_per_slice;
  int qp_bf16;           // DYN: the activation's scale is rounded to bf16
};

// How a weight is stored.
enum Format { kInt8F32, kInt8Bf16, kUint4 };

// 32 consecutive k of one weight row; operand(s): elements 8 s .. 8 s + 7 as an MFMA operand.
template <int FMT>
struct WeightPiece {
  u32x4_t v[2];
  float sc, z;
  __device__ __forceinline__ void clear() { v[0] = v[1] = u32x4_t{0, 0, 0, 0}; sc = z = 0.f; }
  __device__ __forceinline__ u32x4_t operand(int s) const { return int8_operand(v[s >> 1][2 * (s & 1)], v[s >> 1][2 * (s & 1) + 1], sc, z); }
};
template <>
struct WeightPiece<kUint4> {
  u32x4_t codes;
  uint32_t sz;
  __device__ __forceinline__ void clear() { codes = u32x4_t{0, 0, 0, 0}; sz = 0; }
  __device__ __forceinline__ u32x4_t operand(int s) const { return uint4_operand(codes[s], lo_of(sz), hi_of(sz)); }
};

constexpr int kStreamTokens = 16;

// DYN: x arrives as it is and every workgroup fake-quantises it per token into LDS while its first weights are on their way:
// at one token that is 8 - 28 KB read from the cache per workgroup, against a launch of its own (3.8 us and a gap per
// linear: a fifth of a generating layer's time).  A thread holds its share of x, kDynPieces pieces of 8 elements, in
// registers between the extrema and the rounding; a wave's piece lies within one token (one token, or rows of whole pieces).
constexpr int kDynPieces = 4;
constexpr int kDynMaxTokens = 8;

template <int T>  // threads of the workgroup
__device__ __forceinline__ void quantise_tokens(const Int4Args& a, const u32x4_t (&raw)[kDynPieces], uint16_t* xq, float (*ext)[kDynPieces * T / 64]) {
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  constexpr int NW = T / 64;
  const int total = a.M * (a.K >> 3);  // pieces
  auto extrema = [&](int j, float& mn, float& mx) {  // the qparams use min(amin, 0) and max(amax, 0): zero is the neutral start
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      mn = fminf(fminf(mn, lo_of(raw[j][d])), hi_of(raw[j][d]));
      mx = fmaxf(fmaxf(mx, lo_of(raw[j][d])), hi_of(raw[j][d]));
    }
  };
  auto quantise = [&](int j, const TokenQParams& p) {
    const int piece = j * T + t;
    u32x4_t o;
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = pack_pair(token_fq<true>(lo_of(raw[j][d]), p), token_fq<true>(hi_of(raw[j][d]), p));
    if (piece < total) reinterpret_cast<u32x4_t*>(xq)[piece] = o;
  };
  if (a.M == 1) {  // one pair of extrema for the workgroup
    float mn = 0.f, mx = 0.f;
#pragma unroll
    for (int j = 0; j < kDynPieces; ++j)
      if (j * T < total) extrema(j, mn, mx);
    wave_minmax(mn, mx);
    if (lane == 0) {
      ext[0][wave] = mn;
      ext[1][wave] = mx;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      mn = fminf(mn, ext[0][w]);
      mx = fmaxf(mx, ext[1][w]);
    }
    const TokenQParams p = token_qparams(mn, mx, a.qp_bf16 != 0, kF32Eps);
#pragma unroll
    for (int j = 0; j < kDynPieces; ++j)
      if (j * T < total) quantise(j, p);
  } else {
#pragma unroll
    for (int j = 0; j < kDynPieces; ++j) {
      if (j * T >= total) break;
      float mn = 0.f, mx = 0.f;
      extrema(j, mn, mx);
      wave_minmax(mn, mx);
      if (lane == 0) {
        ext[0][j * NW + wave] = mn;
        ext[1][j * NW + wave] = mx;
      }
    }
    __syncthreads();
    const int per_token = a.K >> 9;  // wave pieces per token, at most 64
#pragma unroll
    for (int j = 0; j < kDynPieces; ++j) {
      if (j * T >= total) break;
      const int m = (j * NW + wave) / per_token;  // uniform over the wave
      float mn = 0.f, mx = 0.f;
      if (m < a.M && lane < per_token) {
        mn = ext[0][m * per_token + lane];
        mx = ext[1][m * per_token + lane];
      }
      wave_minmax(mn, mx);
      quantise(j, token_qparams(mn, mx, a.qp_bf16 != 0, kF32Eps));
    }
  }
  __syncthreads();
}

// One wave's stage of a streaming workgroup in LDS: 128 columns of x (MQ groups of four tokens; none where the workgroup
// quantised x itself), of the codes of RT row tiles, and of their scales and zero points.
template <int FMT, int RT, int MQ>
struct StreamStage {
  static constexpr int kX = MQ * 1024;
  static constexpr int kCodes = FMT == kUint4 ? 1024 : 2048;
  static constexpr int kScales = FMT == kInt8F32 ? 512 : FMT == kUint4 ? 256 : 0;  // bf16 scales go to registers
  static constexpr int kBytes = kX + RT * (kCodes + kScales);
};

// RT tiles of 16 weight rows per workgroup (they share a wave's fragments of x), at most MAXW waves (DYN: exactly).  Dynamic
// LDS: DYN: the quantised x; then the waves' stages.  Everything a chunk needs comes by direct-to-LDS loads in row order
// (four neighbouring lanes ask for one row's neighbouring bytes: the address unit takes them together; straight into the
// lanes of an MFMA operand, whose neighbours are different rows, it was what bounded the kernel).
template <int FMT, int RT, int MAXW, bool DYN, int MQ>
__global__ __launch_bounds__(64 * MAXW) void int4_stream_kernel(const Int4Args a) {
#if defined(__HIP_DEVICE_COMPILE__)  // LDS address-space casts
  using S = StreamStage<FMT, RT, DYN ? 0 : MQ>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float ext[2][DYN ? kDynPieces * MAXW : 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int n0 = (int)blockIdx.x * (16 * RT);  // N % 64 == 0: every row of the workgroup exists
  uint16_t* const xq = reinterpret_cast<uint16_t*>(smem);
  const int xq_bytes = DYN ? a.M * a.K * 2 : 0;
  char* const stages = smem + ((xq_bytes + 1023) & ~1023);
  char* const stage = stages + wave * S::kBytes;
  const uint32_t lds = (uint32_t)(uintptr_t)TT_LDS_PTR(stage);
  auto dma16 = [&](uint32_t voff, const void* base, uint32_t at) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(at) : "memory", "m0");
  };
  auto dma4 = [&](uint32_t voff, const void* base, uint32_t at) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(base), "s"(at) : "memory", "m0");
  };
  const int n_chunks = (a.K + 127) >> 7;
  // Piece p of row r goes to slot p ^ (a function of r) such that an operand's 16 lanes read disjoint banks.  int8: 8 pieces
  // a row and chunk, 8 rows an instruction; uint4: 4 and 16; x: 16 and 4.  Pieces beyond K repeat one of the first 32
  // columns (K % 32 == 0: they exist); what they hold is zeroed where it would count.
  float sc_next[RT], z_next[RT];  // bf16 scales
  auto request = [&](int c) {
    const int left = a.K - c * 128;  // columns, at least 32
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int64_t row0 = n0 + 16 * rt;
      if constexpr (FMT == kUint4) {
        const int r = lane >> 2;
        int p = (lane & 3) ^ ((r >> 2) & 3);
        p = 32 * p < left ? p : 0;
        dma16((uint32_t)r * (uint32_t)(a.K >> 1) + 16 * p, a.q + ((row0 * a.K) >> 1) + (int64_t)c * 64, lds + S::kX + rt * S::kCodes);
      } else {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const int r = 8 * d + (lane >> 3);
          int p = (lane & 7) ^ (r >> 1);
          p = 16 * p < left ? p : p & 1;
          dma16((uint32_t)r * (uint32_t)a.K + 16 * p, a.q + row0 * a.K + (int64_t)c * 128, lds + S::kX + rt * S::kCodes + d * 1024);
        }
      }
      if constexpr (FMT == kUint4) {  // [K / g, N]: 16 rows are 64 contiguous bytes; slot i + 16 g
        const int k = c * 128 + (32 * g < left ? 32 * g : 0);
        dma4((uint32_t)(((k >> a.log2_group) * (int64_t)a.N + i) * 4), reinterpret_cast<const uint32_t*>(a.scale) + row0,
             lds + S::kX + RT * S::kCodes + rt * S::kScales);
      } else {
        const int64_t groups = a.K >> a.log2_group;
        if constexpr (FMT == kInt8F32) {  // [N, K / g]; slot 4 row + group of 32
          const int k = c * 128 + (32 * (lane & 3) < left ? 32 * (lane & 3) : 0);
          const uint32_t off = (uint32_t)(((lane >> 2) * groups + (k >> a.log2_group)) * 4);
          dma4(off, reinterpret_cast<const float*>(a.scale) + row0 * groups, lds + S::kX + RT * S::kCodes + rt * S::kScales);
          if (a.zero) dma4(off, reinterpret_cast<const float*>(a.zero) + row0 * groups, lds + S::kX + RT * S::kCodes + rt * S::kScales + 256);
        } else {
          const int64_t at = (row0 + i) * groups + ((c * 128 + (32 * g < left ? 32 * g : 0)) >> a.log2_group);
          sc_next[rt] = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(a.scale)[at]);
          z_next[rt] = a.zero ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(a.zero)[at]) : 0.f;
        }
      }
    }
    if constexpr (!DYN) {
#pragma unroll
      for (int d = 0; d < MQ; ++d) {
        const int r = 4 * d + (lane >> 4), row = r < a.M ? r : a.M - 1;  // rows beyond M repeat the last one: never stored
        int p = (lane & 15) ^ r;
        p = 8 * p < left ? p : p & 3;
        dma16((uint32_t)row * (uint32_t)a.K * 2u + 16 * p, reinterpret_cast<const char*>(a.x) + (int64_t)c * 256, lds + d * 1024);
      }
    }
  };
  int c = wave;
  if constexpr (DYN) {
    // x is asked for ahead of the weights, which then stay in flight while it is quantised; a thread's pieces are brought by
    // its own wave
    const int total = a.M * (a.K >> 3);
#pragma unroll
    for (int j = 0; j < kDynPieces; ++j) {
      const int first = (j * MAXW + wave) * 64;
      if (first < total) dma16((uint32_t)(first + lane < total ? first + lane : first) * 16u, a.x, (uint32_t)(uintptr_t)TT_LDS_PTR(smem) + first * 16);
    }
    if (c < n_chunks) {
      request(c);
      if (FMT == kInt8F32 && a.zero)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * RT) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((FMT == kInt8F32 ? 3 : 2) * RT) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    u32x4_t raw[kDynPieces];
#pragma unroll
    for (int j = 0; j < kDynPieces; ++j) {
      const int piece = j * 64 * MAXW + (int)threadIdx.x;
      raw[j] = u32x4_t{0, 0, 0, 0};
      if (piece < total) raw[j] = reinterpret_cast<const u32x4_t*>(xq)[piece];
    }
    quantise_tokens<64 * MAXW>(a, raw, xq, ext);
  } else {
    if (c < n_chunks) request(c);
  }
  f32x4_t acc[RT][4];  // four chains
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int s = 0; s < 4; ++s) acc[rt][s] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int xr = i & (4 * MQ - 1);  // DYN: tokens beyond M read the first one
  const uint16_t* xrow = xq + (int64_t)(i < a.M ? i : 0) * a.K + 32 * g;
  for (; c < n_chunks; c += nw) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // the stage goes to registers and is asked for again
    WeightPiece<FMT> w[RT];
    u32x4_t xb[4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const char* codes = stage + S::kX + rt * S::kCodes;
      const char* scales = stage + S::kX + RT * S::kCodes + rt * S::kScales;
      if constexpr (FMT == kUint4) {
        w[rt].codes = *reinterpret_cast<const u32x4_t*>(codes + i * 64 + ((g ^ ((i >> 2) & 3)) << 4));
        w[rt].sz = *reinterpret_cast<const uint32_t*>(scales + lane * 4);
      } else {
#pragma unroll
        for (int d = 0; d < 2; ++d) w[rt].v[d] = *reinterpret_cast<const u32x4_t*>(codes + i * 128 + (((2 * g + d) ^ (i >> 1)) << 4));
        if constexpr (FMT == kInt8F32) {
          w[rt].sc = *reinterpret_cast<const float*>(scales + i * 16 + g * 4);
          w[rt].z = a.zero ? *reinterpret_cast<const float*>(scales + 256 + i * 16 + g * 4) : 0.f;
        } else {
          w[rt].sc = sc_next[rt];
          w[rt].z = z_next[rt];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if constexpr (DYN)
        xb[s] = *reinterpret_cast<const u32x4_t*>(xrow + c * 128 + 8 * s);
      else
        xb[s] = *reinterpret_cast<const u32x4_t*>(stage + xr * 256 + (((4 * g + s) ^ xr) << 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (c + nw < n_chunks) request(c + nw);
    if (c * 128 + 32 * g >= a.K) {  // nothing beyond K counts, whatever lies there
#pragma unroll
      for (int s = 0; s < 4; ++s) xb[s] = u32x4_t{0, 0, 0, 0};
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) w[rt].clear();
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
        acc[rt][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[rt].operand(s)),
                                                             __builtin_bit_cast(bf16x8_t, xb[s]), acc[rt][s], 0, 0, 0);
  }
  // partial sums, [tile][lane][v] at the head of each wave's stage, added in wave order by all threads
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) *reinterpret_cast<f32x4_t*>(stage + rt * 1024 + lane * 16) = ((acc[rt][0] + acc[rt][1]) + acc[rt][2]) + acc[rt][3];
  __syncthreads();
  for (int e = threadIdx.x; e < 256 * RT; e += blockDim.x) {
    const int token = (e >> 2) & 15, n = n0 + 16 * (e >> 8) + 4 * ((e >> 6) & 3) + (e & 3);
    if (token >= a.M) continue;
    const char* p = stages + (e >> 8) * 1024 + (e & 255) * 4;
    float o = *reinterpret_cast<const float*>(p);
    if (nw == MAXW) {
#pragma unroll
      for (int q = 1; q < MAXW; ++q) o += *reinterpret_cast<const float*>(p + q * S::kBytes);
    } else {
      for (int q = 1; q < nw; ++q) o += *reinterpret_cast<const float*>(p + q * S::kBytes);
    }
    if (a.bias) o += bf16_bits_to_f32(a.bias[n]);
    a.y[(int64_t)token * a.N + n] = (uint16_t)pack_pair(o, 0.f);
  }
#endif
}

// Eight waves, 64 weight rows, 32 MT tokens; blockIdx = (row tile, token tile, slice of the contraction).  A step is 128 k:
// wave (kg, rg) multiplies the 32 k of its kg by the 32 weight rows of its rg and all tokens; the four kg's sums meet in LDS.
//
// What bounds it: the instructions of the expansion beside the matrix pipes.  Two waves per SIMD (one workgroup per CU at most sizes)
// issue one instruction in 5.5 clocks each; of the 165 of a wave's step at 75 tokens 78 are the expansion's, 6 products, 7 reads of LDS
// and 4 loads.  A step takes 0.5 - 0.6 us, 32 of them on 224 CUs for 14336 x 4096.
//   * Four waves that expanded a fragment for 16-token products, read x from LDS for every 16 rows and went through registers
//     to stage it took 35 us there at 75 tokens, in two slices and their sum; this takes 26 (uint4; int8 42 and 34), 44 and 27
//     at 128, 71 and 54 at 256.
//   * 32 x 32 x 16 products: one read of x from LDS serves 32 weight rows, and up to six other instructions ride under one.
//   * The barrier lies between the two products of a step: with it ahead of both, a stage less was in flight, which three
//     stages (int8 at 128 tokens) do not have to spare: 50 us, 41 now.
template <int FMT, int MT>
struct TileStage {
  static constexpr int kX = MT * 8192;
  static constexpr int kCodeRow = FMT == kUint4 ? 64 : 128;
  static constexpr int kCodes = 64 * kCodeRow;
  static constexpr int kScales = FMT == kUint4 ? 1024 : 2048;
  static constexpr int kBytes = kX + kCodes + kScales;
  static constexpr int kFit = (MT == 1 ? 80 : 160) * 1024 / kBytes, kStages = kFit < 6 ? kFit : 6;  // of 32 tokens two workgroups fit a CU
  static constexpr int kLoads = MT + (FMT == kUint4 ? 1 : 2);  // a wave's loads per step
  static constexpr int kSumRow = 272;  // bytes of a token's 64 partial sums, padded: 8 lanes of a write fall on all banks
  static constexpr int kSums = 4 * 32 * MT * kSumRow;
  static constexpr int kLds = kStages * kBytes > kSums ? kStages * kBytes : kSums;
  static_assert(kStages >= 3 && kLds <= 160 * 1024, "the LDS of a CU");
};

template <int FMT, int MT, bool SPLIT>
__global__ __launch_bounds__(512, 2) void int4_tile_kernel(const Int4Args a) {
#if defined(__HIP_DEVICE_COMPILE__)  // LDS address-space casts
  using S = TileStage<FMT, MT>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wv >> 1, rg = wv & 1;
  const int l31 = lane & 31, h = lane >> 5;
  const int n0 = (int)blockIdx.x * 64;  // N % 64 == 0: every row of the workgroup exists
  const int m0 = (int)blockIdx.y * (32 * MT);
  const int n_chunks = (a.K + 127) >> 7;
  const int t_begin = SPLIT ? (int)blockIdx.z * a.chunks_per_slice : 0;
  const int t_end = SPLIT ? min(t_begin + a.chunks_per_slice, n_chunks) : n_chunks;
  const int groups = a.K >> a.log2_group;

  // ---- loads into the ring.  Piece p (16 bytes) of row r goes to slot p ^ (a function of r) such that an operand's lanes read
  // disjoint banks.  Pieces beyond K repeat one of the step's first 32 columns (K % 32 == 0: they exist); the waves that
  // would multiply them sit the step out.
  const uint32_t ring0 = (uint32_t)(uintptr_t)TT_LDS_PTR(smem);
  uint32_t x_off[MT], c_off;
  auto set_offsets = [&](int left) {
#pragma unroll
    for (int d = 0; d < MT; ++d) {
      const int r = wv * 4 * MT + 4 * d + (lane >> 4);
      int p = (lane & 15) ^ (r & 15);
      p = 8 * p < left ? p : p & 3;
      int row = m0 + r;
      row = row < a.M ? row : a.M - 1;  // tokens beyond M repeat the last one and are never stored
      x_off[d] = (uint32_t)row * (uint32_t)a.K * 2u + 16 * p;
    }
    // uint4: waves 0 - 3 bring the codes and 4 - 7 the scales; int8: all the codes, 0 - 3 the scales and 4 - 7 the zero points
    if constexpr (FMT == kUint4) {
      const int r = (wv & 3) * 16 + (lane >> 2);
      int p = (lane & 3) ^ ((r >> 2) & 3);
      p = 32 * p < left ? p : 0;
      c_off = (uint32_t)r * (uint32_t)(a.K >> 1) + 16 * p;
    } else {
      const int r = wv * 8 + (lane >> 3);
      int p = (lane & 7) ^ ((r >> 1) & 7);
      p = 16 * p < left ? p : p & 1;
      c_off = (uint32_t)r * (uint32_t)a.K + 16 * p;
    }
  };
  set_offsets(128);
  auto dma16 = [&](uint32_t voff, const void* base, uint32_t at) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(at) : "memory", "m0");
  };
  auto dma4 = [&](uint32_t voff, const void* base, uint32_t at) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(base), "s"(at) : "memory", "m0");
  };
  const char* const codes0 = reinterpret_cast<const char*>(a.q) + (((int64_t)n0 * a.K) >> (FMT == kUint4 ? 1 : 0));
  const char* scales0 = reinterpret_cast<const char*>(FMT != kUint4 && wv >= 4 && a.zero ? a.zero : a.scale);
  // bf16 scales and zero points come as the dwords that they lie in (N * K / g is even); zero points may start in the middle of one
  const uint32_t zero_shift = FMT == kInt8Bf16 ? (uint32_t)((uintptr_t)a.zero >> 1) & 1u : 0u;
  const uint32_t my_shift = wv >= 4 ? zero_shift : 0u;
  scales0 -= 2 * my_shift;
  auto issue = [&](int c, uint32_t stage, int d) {  // load d of step c
    const int left = a.K - c * 128;  // columns, at least 32
    if (d < MT) {
      if (d == 0 && left < 128) set_offsets(left);  // the last step
      dma16(x_off[d], reinterpret_cast<const char*>(a.x) + (int64_t)c * 256, ring0 + stage + wv * (MT * 1024) + d * 1024);
    } else if (FMT == kUint4 ? wv < 4 : d == MT) {
      dma16(c_off, codes0 + (int64_t)c * (FMT == kUint4 ? 64 : 128), ring0 + stage + S::kX + wv * 1024);
    } else if constexpr (FMT == kUint4) {  // [K / g, N]; slot 64 (32 of k) + row
      const int k = c * 128 + (32 * (wv & 3) < left ? 32 * (wv & 3) : 0);
      dma4(((uint32_t)(k >> a.log2_group) * (uint32_t)a.N + (uint32_t)(n0 + lane)) * 4u, scales0, ring0 + stage + S::kX + S::kCodes + (wv & 3) * 256);
    } else {  // [N, K / g]; slot 4 row + (32 of k)
      const int kb = lane & 3, k = c * 128 + (32 * kb < left ? 32 * kb : 0);
      const uint32_t e = (uint32_t)(n0 + (wv & 3) * 16 + (lane >> 2)) * (uint32_t)groups + (uint32_t)(k >> a.log2_group);
      const uint32_t off = FMT == kInt8F32 ? e * 4u : ((e + my_shift) & ~1u) * 2u;
      dma4(off, scales0, ring0 + stage + S::kX + S::kCodes + wv * 256);
    }
  };

  // ---- operands.  Lane (l31, h) holds k 32 kg + 16 h + 8 s .. + 7 of row l31 for product s of a step.
  constexpr int kDwords = FMT == kUint4 ? 2 : 4;
  struct Weights {
    uint32_t codes[kDwords];
    float sc, z;
  };
  auto read_weights = [&](int c, uint32_t stage) {
    Weights w;
    const char* codes = smem + stage + (S::kX + (32 * rg + l31) * S::kCodeRow);
    const char* scales = smem + stage + S::kX + S::kCodes;
    if constexpr (FMT == kUint4) {
      const u32x2_t v = *reinterpret_cast<const u32x2_t*>(codes + ((kg ^ ((l31 >> 2) & 3)) << 4) + 8 * h);
      w.codes[0] = v.x;
      w.codes[1] = v.y;
      const uint32_t sz = *reinterpret_cast<const uint32_t*>(scales + (kg * 64 + 32 * rg + l31) * 4);
      w.sc = lo_of(sz);
      w.z = hi_of(sz);
    } else {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(codes + (((2 * kg + h) ^ ((l31 >> 1) & 7)) << 4));
#pragma unroll
      for (int d = 0; d < 4; ++d) w.codes[d] = v[d];
      const char* at = scales + (4 * (32 * rg + l31) + kg) * 4;
      if constexpr (FMT == kInt8F32) {
        w.sc = *reinterpret_cast<const float*>(at);
        w.z = a.zero ? *reinterpret_cast<const float*>(at + 1024) : 0.f;
      } else {
        const uint32_t e = (uint32_t)(n0 + 32 * rg + l31) * (uint32_t)groups + (uint32_t)((c * 128 + 32 * kg) >> a.log2_group);
        const uint32_t s2 = *reinterpret_cast<const uint32_t*>(at), z2 = *reinterpret_cast<const uint32_t*>(at + 1024);
        w.sc = e & 1u ? hi_of(s2) : lo_of(s2);
        w.z = !a.zero ? 0.f : (e + zero_shift) & 1u ? hi_of(z2) : lo_of(z2);
      }
    }
    return w;
  };
  auto expand = [&](const Weights& w, int s) {
    if constexpr (FMT == kUint4) return uint4_operand(w.codes[s], w.sc, w.z);
    else return int8_operand(w.codes[2 * s], w.codes[2 * s + 1], w.sc, w.z);
  };
  int x_at[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) x_at[s] = l31 * 256 + (((4 * kg + 2 * h + s) ^ (l31 & 15)) << 4);
  auto read_x = [&](uint32_t stage, int s, int i) {
    return *reinterpret_cast<const bf16x8_t*>(smem + stage + x_at[s] + i * 8192);
  };
  auto landed = [&](int left) {  // this wave's loads but those of the newest `left` steps, and everybody is here
    if (S::kStages > 5 && left >= 4) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(4 * S::kLoads) : "memory");
    else if (S::kStages > 4 && left >= 3) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * S::kLoads) : "memory");
    else if (S::kStages > 3 && left >= 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * S::kLoads) : "memory");
    else if (left >= 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(S::kLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  };

  f32x16_t acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;
  const int n_steps = t_end - t_begin;
  const int filled = n_steps < S::kStages ? n_steps : S::kStages;
  for (int p = 0; p < filled; ++p) {
#pragma unroll
    for (int d = 0; d < S::kLoads; ++d) issue(t_begin + p, p * S::kBytes, d);
  }
  landed(filled - 1 < S::kStages - 2 ? filled - 1 : S::kStages - 2);
  bf16x8_t xf[2][MT];
  u32x4_t wf[2];
  Weights w = read_weights(t_begin, 0);
#pragma unroll
  for (int i = 0; i < MT; ++i) xf[0][i] = read_x(0, 0, i);
  wf[0] = expand(w, 0);

  // The barrier of step t stands between its two products: by then a wave has the step's operands in registers, so the loads of
  // step t + stages may take its stage, and everybody's loads of step t + 1 have landed.  Beside the first product the weights
  // of the second are expanded, beside the second those of the next step's first.
  uint32_t stage = 0;
  auto step = [&](int t, auto steady) {
    constexpr bool kSteady = decltype(steady)::value;
    const uint32_t here = stage;
    stage = stage == (S::kStages - 1) * S::kBytes ? 0 : stage + S::kBytes;
#pragma unroll
    for (int i = 0; i < MT; ++i) xf[1][i] = read_x(here, 1, i);
    wf[1] = expand(w, 1);
#pragma unroll
    for (int i = 0; i < MT; ++i)
      acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wf[0]), xf[0][i], acc[i], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kSteady) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S::kStages - 2) * S::kLoads) : "memory");
    } else {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      landed(t_end - t - 2 < S::kStages - 2 ? t_end - t - 2 : S::kStages - 2);
    }
    w = read_weights(t + 1, stage);
#pragma unroll
    for (int i = 0; i < MT; ++i) xf[0][i] = read_x(stage, 0, i);
    if constexpr (kSteady) {
#pragma unroll
      for (int d = 0; d < S::kLoads; ++d) issue(t + S::kStages, here, d);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
      acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wf[1]), xf[1][i], acc[i], 0, 0, 0);
    wf[0] = expand(w, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  int t = t_begin;
  for (; t + S::kStages < t_end; ++t) step(t, std::true_type());
  const int tail = a.K & 127;
  const int t_stop = tail != 0 && 32 * kg >= tail && t_end == n_chunks ? t_end - 1 : t_end;
  for (; t < t_stop; ++t) step(t, std::false_type());
  if (t < t_end) landed(0);

  // ---- the four kg's sums meet in LDS, in order
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<f32x4_t*>(smem + (kg * 32 * MT + 32 * i + l31) * S::kSumRow + (32 * rg + 8 * q + 4 * h) * 4) =
          f32x4_t{acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]};
  __syncthreads();
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int token = 32 * j + ((int)threadIdx.x >> 4), quad = threadIdx.x & 15, m = m0 + token;
    if (m >= a.M) continue;
    f32x4_t o = *reinterpret_cast<const f32x4_t*>(smem + token * S::kSumRow + quad * 16);
#pragma unroll
    for (int q = 1; q < 4; ++q) o += *reinterpret_cast<const f32x4_t*>(smem + (q * 32 * MT + token) * S::kSumRow + quad * 16);
    const int nb = n0 + 4 * quad;
    if constexpr (SPLIT) {
      *reinterpret_cast<f32x4_t*>(a.part + ((int64_t)blockIdx.z * a.M + m) * a.N + nb) = o;
    } else {
      if (a.bias) {
        const u32x2_t b = *reinterpret_cast<const u32x2_t*>(a.bias + nb);
        o += f32x4_t{lo_of(b.x), hi_of(b.x), lo_of(b.y), hi_of(b.y)};
      }
      u32x2_t out;
      out.x = pack_pair(o[0], o[1]);
      out.y = pack_pair(o[2], o[3]);
      *reinterpret_cast<u32x2_t*>(a.y + (int64_t)m * a.N + nb) = out;
    }
  }
#endif
}

// y = bf16(sum of the slices in order + bias), four columns per thread
__global__ __launch_bounds__(256) void int4_reduce_kernel(const float* __restrict__ part, int slices, int64_t quads, int nq,
                                                          const uint16_t* __restrict__ bias, uint16_t* __restrict__ y) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= quads) return;
  const f32x4_t* p = reinterpret_cast<const f32x4_t*>(part) + e;
  f32x4_t o = p[0];
  for (int s = 1; s < slices; ++s) o += p[s * quads];
  if (bias) {
    const u32x2_t b = reinterpret_cast<const u32x2_t*>(bias)[e % nq];
    o += f32x4_t{lo_of(b.x), hi_of(b.x), lo_of(b.y), hi_of(b.y)};
  }
  u32x2_t out;
  out.x = pack_pair(o[0], o[1]);
  out.y = pack_pair(o[2], o[3]);
  reinterpret_cast<u32x2_t*>(y)[e] = out;
}

constexpr int kMaxTokens = 256;
constexpr int kMinRows = 256;

// 32-token tiles per workgroup: as few rows of padding as token tiles of at most 128 allow
int tile_mt(int64_t M) {
  const int64_t tiles = (M + 127) / 128;
  return (int)((M + 32 * tiles - 1) / (32 * tiles));
}

struct Slicing {
  int slices, chunks;
};
// Slices of the contraction, by the time they take (us, fitted to all slicings of ten layers at 32 - 256 tokens): a round of
// workgroups 4.2 and 0.43 + 0.05 per 32 tokens a step; the sum 1.8, 0.15 a slab and 0.65 a MB of slabs.  One workgroup fits a CU, of 32
// tokens two, which take 1.5 times as long together.  75 tokens: 14336 x 4096 (224 row tiles) 26 whole, 33 in two slices, 4096 x 14336
// (64) 75 whole, 28 in four, 33 in eight; 1024 x 4096 (16) 23 whole, 11 in eight, 13 in sixteen.  Beyond 512 workgroups only the slabs
// grow.  A wave adds a quarter of its slice in one chain, which is at most as long as with 512 workgroups of one chain per slice.
Slicing slicing(int64_t M, int64_t N, int64_t K) {
  const int64_t n_chunks = (K + 127) / 128;
  const int mt = tile_mt(M);
  const int64_t wgs = (N / 64) * ((M + 32 * mt - 1) / (32 * mt));
  int64_t fine = wgs < 512 ? 512 / wgs : 1;
  fine = std::min({fine, std::max<int64_t>(n_chunks / 4, 1), int64_t(16)});
  const int64_t longest = 4 * ((n_chunks + fine - 1) / fine);
  Slicing best = {};
  double best_us = 0;
  for (int64_t s = 1; s <= 16 && s <= n_chunks && (s == 1 || wgs * s <= 512); ++s) {
    const int64_t chunks = (n_chunks + s - 1) / s, slices = (n_chunks + chunks - 1) / chunks;
    if (chunks > longest) continue;
    const double rounds = mt > 1 || wgs * slices <= 256 ? (double)((wgs * slices + 255) / 256) : 1.5 * ((wgs * slices + 511) / 512);
    double us = rounds * (4.2 + chunks * (0.43 + 0.05 * mt));
    if (slices > 1) us += 1.8 + slices * (0.15 + 0.65e-6 * 4 * M * N);
    if (best.slices == 0 || us < best_us) {
      best = {(int)slices, (int)chunks};
      best_us = us;
    }
  }
  return best;
}

template <int FMT, int MT, bool SPLIT>
int launch_tile(const Int4Args& a, dim3 grid, hipStream_t s) {
  constexpr int kLds = TileStage<FMT, MT>::kLds;
  static bool attr_set[64] = {};  // the LDS limit is a per-device attribute of the function
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (dev < 0 || !attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&int4_tile_kernel<FMT, MT, SPLIT>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) return fail(TTAMD_ELAUNCH, "int4_linear: cannot reserve %d bytes of LDS: %s", kLds, hipGetErrorString(e));
    if (dev >= 0) attr_set[dev] = true;
  }
  int4_tile_kernel<FMT, MT, SPLIT><<<grid, dim3(512), kLds, s>>>(a);
  return check_launch("int4_linear");
}
template <int FMT, bool SPLIT>
int launch_tile(const Int4Args& a, int mt, dim3 grid, hipStream_t s) {
  switch (mt) {
    case 1: return launch_tile<FMT, 1, SPLIT>(a, grid, s);
    case 2: return launch_tile<FMT, 2, SPLIT>(a, grid, s);
    case 3: return launch_tile<FMT, 3, SPLIT>(a, grid, s);
    default: return launch_tile<FMT, 4, SPLIT>(a, grid, s);
  }
}

template <int FMT, int RT, int MAXW, bool DYN, int MQ>
int launch_stream(const Int4Args& a, hipStream_t s) {
  using S = StreamStage<FMT, RT, DYN ? 0 : MQ>;
  const int n_chunks = (a.K + 127) >> 7, waves = DYN || n_chunks > MAXW ? MAXW : n_chunks;
  const int head = DYN ? (a.M * a.K * 2 + 1023) & ~1023 : 0;
  constexpr int kMost = (DYN ? 64 * MAXW * kDynPieces * 16 + 1023 : 0) + MAXW * S::kBytes;
  static_assert(kMost + 2 * 4 * kDynPieces * MAXW <= 160 * 1024, "the LDS of a CU");
  static_assert(S::kBytes >= RT * 1024, "the partial sums fit a stage");
  static bool attr_set[64] = {};  // the LDS limit is a per-device attribute of the function
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (dev < 0 || !attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&int4_stream_kernel<FMT, RT, MAXW, DYN, MQ>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kMost);
    if (e != hipSuccess) return fail(TTAMD_ELAUNCH, "int4_linear: cannot reserve %d bytes of LDS: %s", kMost, hipGetErrorString(e));
    if (dev >= 0) attr_set[dev] = true;
  }
  int4_stream_kernel<FMT, RT, MAXW, DYN, MQ><<<dim3(a.N / (16 * RT)), dim3(64 * waves), head + waves * S::kBytes, s>>>(a);
  return check_launch("int4_linear");
}
template <int FMT, int RT, int MAXW>
int launch_stream(const Int4Args& a, bool dyn, hipStream_t s) {
  if constexpr (FMT != kUint4) {
    if (dyn) return launch_stream<FMT, RT, MAXW, true, 1>(a, s);
  }
  return a.M <= 4 ? launch_stream<FMT, RT, MAXW, false, 1>(a, s) : launch_stream<FMT, RT, MAXW, false, 4>(a, s);
}

// Waves of the int8 launch of at most 16 tokens, and whether it can quantise these activations itself: they fit the pieces
// its threads hold, and no wave's piece crosses a row.
int int8_stream_waves(int64_t N, int64_t K) { return N >= 2048 && N < 8192 && K >= 4096 ? 16 : 8; }
bool quantises_in_stream(int64_t M, int64_t N, int64_t K) {
  return M <= kDynMaxTokens && (M == 1 ? K <= int8_stream_waves(N, K) * 64 * kDynPieces * 8 : K % 512 == 0 && M * K <= 16384);
}

// dyn: x is not quantised yet (quantises_in_stream holds)
template <int FMT>
int launch(Int4Args& a, bool dyn, void* workspace, size_t workspace_bytes, hipStream_t s) {
  if (a.M <= kStreamTokens) {
    // Measured (weights from HBM, us, launch gap included).  The waves fix the order of a row's sums and depend on the layer
    // alone.  int8 at one token, eight and sixteen: 4096 x 4096 8.5 and 8.0, 4096 x 14336 17.5 and 16.5, but 1024 x 4096 6.1 and 6.6; a wide
    // layer has workgroups enough for eight, and two row tiles from two tokens on (14336 x 4096 at 1 / 4 tokens: one 17.7 / 26.1,
    // two 17.5 / 20.6; 8192 x 2048 at one 7.0 and 7.6).  uint4: narrow layers sixteen (4096 x 14336 16.4 and 15.3), wide eight (9728 x 3584
    // 11.5 and 15.7; both pairs with an expansion of 60 instructions, with that of 37 13.5 and 10.3).
    const bool wide = a.N >= 8192;
    if constexpr (FMT == kUint4) {
      return wide ? launch_stream<FMT, 1, 8>(a, dyn, s) : launch_stream<FMT, 1, 16>(a, dyn, s);
    } else {
      if (wide && a.M > 1) return launch_stream<FMT, 2, 8>(a, dyn, s);
      return int8_stream_waves(a.N, a.K) == 16 ? launch_stream<FMT, 1, 16>(a, dyn, s) : launch_stream<FMT, 1, 8>(a, dyn, s);
    }
  }
  const Slicing sl = slicing(a.M, a.N, a.K);
  const int mt = tile_mt(a.M);
  const dim3 grid(a.N / 64, (a.M + 32 * mt - 1) / (32 * mt), sl.slices);
  a.chunks_per_slice = sl.chunks;
  if (sl.slices == 1) return launch_tile<FMT, false>(a, mt, grid, s);
  const size_t need = (size_t)sl.slices * a.M * a.N * sizeof(float);
  if (!workspace || workspace_bytes < need)
    return fail(TTAMD_EWORKSPACE, "int4_linear: workspace of %zu bytes, %zu needed", workspace_bytes, need);
  TT_REQUIRE(aligned16(workspace), "int4_linear: the workspace must be 16-byte aligned");
  a.part = reinterpret_cast<float*>(workspace);
  if (int rc = launch_tile<FMT, true>(a, mt, grid, s)) return rc;
  const int64_t quads = (int64_t)a.M * a.N / 4;
  int4_reduce_kernel<<<dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s>>>(a.part, sl.slices, quads, a.N / 4, a.bias, a.y);
  return check_launch("int4_linear: reduction");
}

int check_args(const void* x, const void* q, const void* scale, const void* y, int64_t M, int64_t N, int64_t K, int group_size) {
  TT_REQUIRE(x && q && scale && y, "int4_linear: x, q, the scales and y must be non-null");
  TT_REQUIRE(aligned16(x) && aligned16(q) && aligned16(scale) && aligned16(y), "int4_linear: pointers must be 16-byte aligned");
  if (!ttamd_int4_linear_applies(M, N, K, group_size))
    return fail(TTAMD_EUNSUPPORTED, "int4_linear: M = %lld, N = %lld, K = %lld, group_size = %d is not served", (long long)M,
                (long long)N, (long long)K, group_size);
  return TTAMD_OK;
}

int log2_of(int v) {
  int l = 0;
  while ((1 << l) < v) ++l;
  return l;
}

}  // namespace
}  // namespace ttamd

using namespace ttamd;

extern "C" int ttamd_int4_linear_applies(int64_t M, int64_t N, int64_t K, int group_size) {
  return M > 0 && M <= kMaxTokens && N >= kMinRows && N % 64 == 0 && K > 0 && K % 32 == 0 && group_size >= 32 &&
         is_pow2(group_size) && K % group_size == 0 && N * K < (int64_t(1) << 31);
}

extern "C" size_t ttamd_int4_linear_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= kStreamTokens || M > kMaxTokens || N < 64 || K <= 0) return 0;
  const Slicing sl = slicing(M, N, K);
  return sl.slices > 1 ? (size_t)sl.slices * M * N * sizeof(float) : 0;
}

extern "C" int ttamd_int8_group_linear_bf16(const void* x, const int8_t* q, const void* scale, const void* zero_point,
                                            int qparam_dtype, int group_size, const void* bias, void* y, int64_t M, int64_t N,
                                            int64_t K, void* workspace, size_t workspace_bytes, void* stream) {
  if (int rc = check_args(x, q, scale, y, M, N, K, group_size)) return rc;
  TT_REQUIRE(qparam_dtype == TTAMD_BF16 || qparam_dtype == TTAMD_F32, "int8_group_linear: unknown qparam dtype code %d", qparam_dtype);
  Int4Args a = {reinterpret_cast<const uint16_t*>(x), reinterpret_cast<const uint8_t*>(q), scale, zero_point,
                reinterpret_cast<const uint16_t*>(bias), reinterpret_cast<uint16_t*>(y), nullptr, (int)M, (int)N, (int)K,
                log2_of(group_size), 0, 0};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return qparam_dtype == TTAMD_BF16 ? launch<kInt8Bf16>(a, false, workspace, workspace_bytes, s)
                                    : launch<kInt8F32>(a, false, workspace, workspace_bytes, s);
}

namespace {
size_t quantised_bytes(int64_t M, int64_t N, int64_t K) {
  return quantises_in_stream(M, N, K) ? 0 : ((size_t)M * K * 2 + 255) / 256 * 256;
}
}  // namespace

extern "C" size_t ttamd_int8_dynamic_linear_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || M > kMaxTokens || N < 64 || K <= 0) return 0;
  return quantised_bytes(M, N, K) + ttamd_int4_linear_workspace_bytes(M, N, K);
}

extern "C" int ttamd_int8_dynamic_linear_bf16(const void* x, const int8_t* q, const void* scale, const void* zero_point,
                                              int qparam_dtype, int group_size, const void* bias, void* y, int64_t M, int64_t N,
                                              int64_t K, void* workspace, size_t workspace_bytes, void* stream) {
  if (int rc = check_args(x, q, scale, y, M, N, K, group_size)) return rc;
  TT_REQUIRE(qparam_dtype == TTAMD_BF16 || qparam_dtype == TTAMD_F32, "int8_dynamic_linear: unknown qparam dtype code %d", qparam_dtype);
  const size_t head = quantised_bytes(M, N, K), need = ttamd_int8_dynamic_linear_workspace_bytes(M, N, K);
  if (need > 0 && (!workspace || workspace_bytes < need))
    return fail(TTAMD_EWORKSPACE, "int8_dynamic_linear: workspace of %zu bytes, %zu needed", workspace_bytes, need);
  TT_REQUIRE(need == 0 || aligned16(workspace), "int8_dynamic_linear: the workspace must be 16-byte aligned");
  if (head > 0) {
    if (int rc = ttamd_fq_per_token_int8_asym(x, TTAMD_BF16, M, K, qparam_dtype, workspace, nullptr, nullptr, stream)) return rc;
    return ttamd_int8_group_linear_bf16(workspace, q, scale, zero_point, qparam_dtype, group_size, bias, y, M, N, K,
                                        reinterpret_cast<char*>(workspace) + head, workspace_bytes - head, stream);
  }
  Int4Args a = {reinterpret_cast<const uint16_t*>(x), reinterpret_cast<const uint8_t*>(q), scale, zero_point,
                reinterpret_cast<const uint16_t*>(bias), reinterpret_cast<uint16_t*>(y), nullptr, (int)M, (int)N, (int)K,
                log2_of(group_size), 0, qparam_dtype == TTAMD_BF16 ? 1 : 0};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return qparam_dtype == TTAMD_BF16 ? launch<kInt8Bf16>(a, true, nullptr, 0, s) : launch<kInt8F32>(a, true, nullptr, 0, s);
}

extern "C" int ttamd_uint4_group_linear_bf16(const void* x, const uint8_t* q, const void* scales_and_zeros, int group_size,
                                             const void* bias, void* y, int64_t M, int64_t N, int64_t K, void* workspace,
                                             size_t workspace_bytes, void* stream) {
  if (int rc = check_args(x, q, scales_and_zeros, y, M, N, K, group_size)) return rc;
  Int4Args a = {reinterpret_cast<const uint16_t*>(x), q, scales_and_zeros, nullptr, reinterpret_cast<const uint16_t*>(bias),
                reinterpret_cast<uint16_t*>(y), nullptr, (int)M, (int)N, (int)K, log2_of(group_size), 0, 0};
  return launch<kUint4>(a, false, workspace, workspace_bytes, reinterpret_cast<hipStream_t>(stream));
}
