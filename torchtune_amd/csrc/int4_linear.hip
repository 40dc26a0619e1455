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
//    bytes of its weight rows).  Four waves own 64 weight rows between them and share 128-wide chunks of up to 128
//    tokens through a double LDS buffer; a weight fragment is expanded once per 128 tokens.  Launches of few tiles cut
//    the contraction into slices (fp32 slabs, added in slice order by int4_reduce_kernel).
//
// Measured against dequantise + library GEMM (us, weights from HBM, launch gaps included; int8 / uint4):
//   14336 x 4096:  1 token 60 / 60 -> 17.7 / 16.1, 16 tokens 59 / 60 -> 25 / 17.8, 75 tokens 63 / 65 -> 38 / 33, 256 tokens 83 / 82 -> 67 / 69
//   4096 x 14336:  1 token 58 / 58 -> 16.5 / 15.3, 75 tokens 79 / 78 -> 38 / 32, 256 tokens 93 / 92 -> 74 / 66
//   1024 x 4096:   1 token 20 / 20 -> 6.1 / 5.9, 256 tokens 21 / 21 -> 17 / 16
// (at most 16 tokens with loads straight into the MFMA lanes and one wave's sum at the end: 26.4 / 19.0, 21.9 / 19.5 and 9.0 / 7.3 at
// one token; a read of the same bytes takes 14 / 6.5).  Above 256 tokens the two m-tiles' expansion and their slabs cost what
// the dense copy costs, and the library's larger tiles win.
#include "common.h"
#include "fq_math.h"
#include "nf4_math.h"

#define TT_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

namespace ttamd {
namespace {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pack_pair(float lo, float hi) {
  bf16x2_t v;
  v.x = (__bf16)lo;
  v.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float lo_of(uint32_t d) { return bits_f32(d << 16); }
__device__ __forceinline__ float hi_of(uint32_t d) { return bits_f32(d & 0xffff0000u); }

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

// 32 consecutive k of one weight row, as loaded.
template <int FMT>
struct WeightPiece;

template <>
struct WeightPiece<kUint4> {
  u32x4_t codes;
  uint32_t sz;
  __device__ __forceinline__ void clear() { codes = u32x4_t{0, 0, 0, 0}; sz = 0; }
  __device__ __forceinline__ void load(const Int4Args& a, int n, int k) {
    codes = *reinterpret_cast<const u32x4_t*>(a.q + (((int64_t)n * a.K + k) >> 1));
    sz = reinterpret_cast<const uint32_t*>(a.scale)[(int64_t)(k >> a.log2_group) * a.N + n];
  }
  // elements 8 s .. 8 s + 7 as an MFMA operand: bf16(bf16((q - 8) * scale) + zero).  The first product is that of 16 (q - 8), a
  // byte with the nibble on top, and scale / 16, both exact (8 * scale, which a fused multiply-add would subtract, overflows
  // for scales above 2^125 whose small multiples do not).
  __device__ __forceinline__ u32x4_t operand(int s) const {
    const float sc = lo_of(sz) * 0.0625f, z = hi_of(sz);
    const uint32_t c = codes[s] ^ 0x88888888u, high = c & 0xf0f0f0f0u, low = (c << 4) & 0xf0f0f0f0u;
    u32x4_t w;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const uint32_t p = pack_pair((float)(int8_t)(high >> (8 * b)) * sc, (float)(int8_t)(low >> (8 * b)) * sc);
      w[b] = pack_pair(lo_of(p) + z, hi_of(p) + z);
    }
    return w;
  }
};

template <bool QP_BF16>
struct Int8Piece {
  u32x4_t v[2];
  float sc, z;
  __device__ __forceinline__ void clear() { v[0] = v[1] = u32x4_t{0, 0, 0, 0}; sc = z = 0.f; }
  __device__ __forceinline__ void load(const Int4Args& a, int n, int k) {
    const u32x4_t* p = reinterpret_cast<const u32x4_t*>(a.q + (int64_t)n * a.K + k);
    v[0] = p[0];
    v[1] = p[1];
    const int64_t gi = (int64_t)n * (a.K >> a.log2_group) + (k >> a.log2_group);
    if constexpr (QP_BF16) {
      sc = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(a.scale)[gi]);
      z = a.zero ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(a.zero)[gi]) : 0.f;
    } else {
      sc = reinterpret_cast<const float*>(a.scale)[gi];
      z = a.zero ? reinterpret_cast<const float*>(a.zero)[gi] : 0.f;
    }
  }
  __device__ __forceinline__ u32x4_t operand(int s) const {  // bf16((q - zero) * scale)
    u32x4_t w;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t two = v[s >> 1][2 * (s & 1) + (d >> 1)] >> (16 * (d & 1));
      w[d] = pack_pair(((float)(int8_t)(two & 0xffu) - z) * sc, ((float)(int8_t)((two >> 8) & 0xffu) - z) * sc);
    }
    return w;
  }
};
template <>
struct WeightPiece<kInt8F32> : Int8Piece<false> {};
template <>
struct WeightPiece<kInt8Bf16> : Int8Piece<true> {};

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

// Four waves, 64 weight rows, 16 MT tokens; blockIdx = (row tile, token tile, slice of the contraction).
template <int FMT, int MT, bool SPLIT>
__global__ __launch_bounds__(256) void int4_tile_kernel(const Int4Args a) {
  // 128 k of 16 MT tokens: token r's 16-byte piece p lies in slot p ^ (r % 16), so that the 16 lanes of a fragment read
  // (16 tokens, one piece each) fall on disjoint banks
  __shared__ u32x4_t xs[2][MT * 16 * 16];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int n = (int)blockIdx.x * 64 + 16 * wave + i;  // N % 64 == 0
  const int m0 = (int)blockIdx.y * (16 * MT);
  const int n_chunks = (a.K + 127) >> 7;
  const int c_first = SPLIT ? (int)blockIdx.z * a.chunks_per_slice : 0;
  const int c_end = SPLIT ? min(c_first + a.chunks_per_slice, n_chunks) : n_chunks;

  // thread t stages piece t % 16 of tokens t / 16 + 16 j
  const int piece = t & 15, row = t >> 4;
  const uint16_t* xsrc[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    int m = m0 + 16 * j + row;
    m = m < a.M ? m : a.M - 1;  // tokens beyond M repeat the last one and are never stored
    xsrc[j] = a.x + (int64_t)m * a.K + 8 * piece;
  }
  const int slot = row * 16 + (piece ^ row);

  f32x4_t acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t xr[MT];
  WeightPiece<FMT> w;
  auto request = [&](int c) {
    const int k = c * 128 + 32 * g;
    if (k < a.K)
      w.load(a, n, k);
    else
      w.clear();
    const bool in = c * 128 + 8 * piece < a.K;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      xr[j] = u32x4_t{0, 0, 0, 0};
      if (in) xr[j] = *reinterpret_cast<const u32x4_t*>(xsrc[j] + c * 128);
    }
  };
  request(c_first);
#pragma unroll
  for (int j = 0; j < MT; ++j) xs[0][j * 256 + slot] = xr[j];
  __syncthreads();
  int buf = 0;
  for (int c = c_first; c < c_end; ++c) {
    const WeightPiece<FMT> wc = w;
    const bool more = c + 1 < c_end;
    if (more) request(c + 1);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bf16x8_t wf = __builtin_bit_cast(bf16x8_t, wc.operand(s));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            wf, __builtin_bit_cast(bf16x8_t, xs[buf][mt * 256 + i * 16 + ((4 * g + s) ^ i)]), acc[mt], 0, 0, 0);
    }
    buf ^= 1;
    if (more) {
#pragma unroll
      for (int j = 0; j < MT; ++j) xs[buf][j * 256 + slot] = xr[j];
    }
    __syncthreads();
  }
  const int nb = (int)blockIdx.x * 64 + 16 * wave + 4 * g;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + 16 * mt + i;
    if (m >= a.M) continue;
    if constexpr (SPLIT) {
      *reinterpret_cast<f32x4_t*>(a.part + ((int64_t)blockIdx.z * a.M + m) * a.N + nb) = acc[mt];
    } else {
      f32x4_t o = acc[mt];
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

// 16-token tiles per workgroup: as few rows of padding as the instantiated sizes allow (75 tokens on 14336 x 4096 int8: five
// tiles 38 us, eight 48 us)
int tile_mt(int64_t M) {
  const int64_t wg_rows = (M + 127) / 128;
  const int mt = (int)((M + 16 * wg_rows - 1) / (16 * wg_rows));
  return mt <= 2 ? 2 : (mt == 7 ? 8 : mt);
}

struct Slicing {
  int slices, chunks;
};
Slicing slicing(int64_t M, int64_t N, int64_t K) {
  const int64_t n_chunks = (K + 127) / 128;
  const int64_t wgs = (N / 64) * ((M + 16 * tile_mt(M) - 1) / (16 * tile_mt(M)));
  // two workgroups per CU and not one more: 64 tokens on 14336 x 4096 (224 row tiles, us, int8) 43 with one slice, 34 with
  // two, 36 with three, 38 with four; on 4096 x 14336 (64 row tiles) 40 / 34 / 37 with four / eight / sixteen
  int64_t s = wgs < 512 ? 512 / wgs : 1;
  const int64_t most = n_chunks / 4 > 1 ? n_chunks / 4 : 1;
  s = s < most ? s : most;
  s = s < 16 ? s : 16;
  const int64_t chunks = (n_chunks + s - 1) / s;
  return {(int)((n_chunks + chunks - 1) / chunks), (int)chunks};
}

template <int FMT, bool SPLIT>
void launch_tile(const Int4Args& a, int mt, dim3 grid, hipStream_t s) {
  const dim3 block(256);
  switch (mt) {
    case 2: int4_tile_kernel<FMT, 2, SPLIT><<<grid, block, 0, s>>>(a); break;
    case 3: int4_tile_kernel<FMT, 3, SPLIT><<<grid, block, 0, s>>>(a); break;
    case 4: int4_tile_kernel<FMT, 4, SPLIT><<<grid, block, 0, s>>>(a); break;
    case 5: int4_tile_kernel<FMT, 5, SPLIT><<<grid, block, 0, s>>>(a); break;
    case 6: int4_tile_kernel<FMT, 6, SPLIT><<<grid, block, 0, s>>>(a); break;
    default: int4_tile_kernel<FMT, 8, SPLIT><<<grid, block, 0, s>>>(a); break;
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
    // 11.5 and 15.7).
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
  const dim3 grid(a.N / 64, (a.M + 16 * mt - 1) / (16 * mt), sl.slices);
  a.chunks_per_slice = sl.chunks;
  if (sl.slices == 1) {
    launch_tile<FMT, false>(a, mt, grid, s);
    return check_launch("int4_linear");
  }
  const size_t need = (size_t)sl.slices * a.M * a.N * sizeof(float);
  if (!workspace || workspace_bytes < need)
    return fail(TTAMD_EWORKSPACE, "int4_linear: workspace of %zu bytes, %zu needed", workspace_bytes, need);
  TT_REQUIRE(aligned16(workspace), "int4_linear: the workspace must be 16-byte aligned");
  a.part = reinterpret_cast<float*>(workspace);
  launch_tile<FMT, true>(a, mt, grid, s);
  if (int rc = check_launch("int4_linear")) return rc;
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
