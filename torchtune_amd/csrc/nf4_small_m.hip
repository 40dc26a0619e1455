// y = x . D(W)^T (+ bias) + scale . h . lora_b^T, times an optional column scale, for a handful of tokens (M <= 64):
// the decode / evaluation regime of linear_nf4 and LoRALinear.forward (torchtune/modules/peft/lora.py:128-147,
// torchtune/modules/low_precision/nf4_linear.py:56-70).
//
// With so few rows the work is streaming the packed weight once: 0.5625 bytes per weight element against 2 for a
// dense bf16 weight.  A workgroup owns 16 or 32 weight rows and the whole contraction, expands the codes in registers
// exactly as the large-M kernel does (byte -> pair of code points from an LDS table, times the fp32 block scaler, one rounding to
// bf16 - the bits of ttamd_nf4_dequantize) and feeds v_mfma_f32_16x16x32_bf16 with the weight rows as the row operand
// and 16-token tiles of x as the column operand.  A lane reads 16 contiguous bytes of codes (32 elements of
// its row: the four lane groups of a row cover one 64-byte piece) and uses one dword of them per MFMA; x is small and
// comes from the cache.  The waves' partial sums meet in LDS in a fixed order.
//
//  * nf4_few_kernel (at most 16 tokens, generation): the waves take 128-wide chunks of K in turn, one chunk in flight each while
//    the one before it is multiplied (more in flight gained nothing).  What bounded its first form was neither HBM nor
//    arithmetic but the address unit - operands loaded straight into MFMA lanes, where neighbouring lanes are different rows,
//    cost it 64 cycles a load instead of 16, and a block scaler's load as much as its 32 codes' - and one wave's sum over
//    the others at the end (1.3 us).  Now codes, x and lora_a come by direct-to-LDS loads in row order, a workgroup's
//    scalers in one pass ahead of the loop, the table holds fp16 pairs (a code point is exact in fp16), which the multiply
//    converts on the way, and every thread finishes outputs.  The hidden product h = x . lora_a^T can ride along as
//    further row tiles of the same loop, where that beats a launch of its own.
//    us, weights from HBM, hidden product included, before -> now at 1 / 13 tokens: 4096 x 4096 12.5 / 14.2 -> 6.7 / 7.6, 14336 x 4096 21.3 /
//    25.7 -> 14.9 / 16.7, 4096 x 14336 22.1 / 30.8 -> 15.6 / 20.4, 2048 x 2048 9.1 / 11.1 -> 5.4 / 5.9, gate / up pair of 14336 x 4096 38.0 / 43.1 ->
//    26.6 / 31.2.  A read of the same bytes in the same row pieces takes 3.1, 6.3, 6.6 and (the pair) 10.3: the pair is bound by
//    the expansion (VALU 10.9 us, LDS 11.7 of 22 us busy without the hidden product).
//  * nf4_small_m_kernel (17 - 64 tokens): groups of U chunks per wave, two or four token tiles.
#include "common.h"
#include "group.h"
#include "nf4_math.h"
#include "swiglu_math.h"

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

struct SmallMArgs {
  const uint16_t* x;       // [M, K] bf16
  const uint8_t* codes;    // [N, K/2]
  const float* bscal;      // [N, K/64]
  const uint16_t* h;       // [M, R] bf16 (rows ldh elements apart) or null
  const uint16_t* lora_a;  // [R, K] bf16 where the launch forms h itself
  uint16_t* h_out;         // and where it leaves it (rows ldh elements apart), or null
  const uint16_t* lora_b;  // [N, R] bf16 or null
  const uint16_t* bias;    // [N] bf16 or null
  const uint16_t* cscale;  // [N] bf16 or null
  uint16_t* y;             // [M, N] bf16
  int M, N, K, R, ldh;
  float lscale;
};
// The layers of one launch: they share x, M and K (projections of a common input); workgroups [wg_end[i - 1], wg_end[i])
// work on layer i.
struct SmallMGroup {
  SmallMArgs m[kGroupMax];
  int wg_end[kGroupMax];
  int n;
};

constexpr int kSmMaxWaves = 16;

// U chunks (128 elements of K each) of RT 16-row tiles: what one wave has in flight.
template <int RT, int U>
struct WeightFrag {
  u32x4_t cd[U][RT];  // 32 codes of this lane's row per chunk
  float sc[U][RT];    // the block scaler of those 32 elements
};

// TAIL: the lane may lie beyond K (the last chunk of a K that is an odd multiple of 64 is half a chunk).
template <int RT, int U, bool TAIL>
__device__ __forceinline__ void load_weights(WeightFrag<RT, U>& f, const uint8_t* crow, const float* srow, int64_t ctile,
                                             int64_t stile, int c0, bool valid) {
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if (TAIL && !valid) {
        f.cd[u][rt] = u32x4_t{0, 0, 0, 0};
        f.sc[u][rt] = 0.f;
      } else {
        f.cd[u][rt] = *reinterpret_cast<const u32x4_t*>(crow + rt * ctile + (int64_t)(c0 + u) * 64);
        f.sc[u][rt] = srow[rt * stile + 2 * (c0 + u)];
      }
    }
}

template <int MT, int RT, int U, int NACC, bool TAIL>
__device__ __forceinline__ void multiply(const WeightFrag<RT, U>& f, const float2* lut, const uint16_t* const (&xrow)[MT], int c0,
                                         bool valid, f32x4_t (&acc)[MT][RT][NACC]) {
  u32x4_t xb[U][4][MT];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if (TAIL && !valid)
          xb[u][s][mt] = u32x4_t{0, 0, 0, 0};
        else
          xb[u][s][mt] = *reinterpret_cast<const u32x4_t*>(xrow[mt] + (c0 + u) * 128 + 8 * s);
      }
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        u32x4_t wf;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const float2 p = lut[(f.cd[u][rt][s] >> (8 * b)) & 0xffu];
          wf[b] = pack_pair(p.x * f.sc[u][rt], p.y * f.sc[u][rt]);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[mt][rt][s % NACC] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, wf), __builtin_bit_cast(bf16x8_t, xb[u][s][mt]), acc[mt][rt][s % NACC], 0, 0, 0);
      }
}

// One NF4 code as fp32 without touching memory (a chain of selects over the sixteen constants).
__device__ __forceinline__ float nf4_code_value(int k) {
  constexpr float tab[16] = TT_NF4_TABLE;
  float v = tab[0];
#pragma unroll
  for (int j = 1; j < 16; ++j) v = k == j ? tab[j] : v;
  return v;
}

// MT 16-token tiles of x, RT 16-row tiles of W per workgroup, U chunks of K in flight per wave, at most MAXW waves (the
// register budget of a lane follows from it: the four-wave shapes hold more tiles per lane).
template <int MT, int RT, int U, int MAXW>
__global__ __launch_bounds__(64 * MAXW) void nf4_small_m_kernel(const SmallMGroup grp) {
  int which = 0;  // uniform over the workgroup
#pragma unroll
  for (int q = 0; q < kGroupMax - 1; ++q)
    if (q < grp.n - 1 && (int)blockIdx.x >= grp.wg_end[q]) which = q + 1;
  const SmallMArgs& a = grp.m[which];
  const int wg = (int)blockIdx.x - (which ? grp.wg_end[which - 1] : 0);
  constexpr int NACC = MT * RT == 2 ? 2 : 1;  // independent MFMA chains per lane: at least four
  __shared__ float2 lut[256];
  extern __shared__ float red[];  // [waves - 1][MT * RT * 4][64]
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nw = blockDim.x >> 6;
  const int i = lane & 15, g = lane >> 4;

  const int K = a.K;
  const int n0 = wg * (16 * RT);  // N % (16 RT) == 0: every row of the workgroup exists
  const uint8_t* crow = a.codes + (((int64_t)(n0 + i) * K) >> 1) + 16 * g;
  const float* srow = a.bscal + (int64_t)(n0 + i) * (K >> 6) + (g >> 1);
  const int64_t ctile = (int64_t)8 * K, stile = (int64_t)16 * (K >> 6);  // one 16-row tile further on
  const uint16_t* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    int m = 16 * mt + i;
    m = m < a.M ? m : a.M - 1;  // rows beyond M repeat the last one and are never stored
    xrow[mt] = a.x + (int64_t)m * K + 32 * g;
  }
  f32x4_t acc[MT][RT][NACC];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int q = 0; q < NACC; ++q) acc[mt][rt][q] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // Groups of U whole chunks go round the waves; what is left (fewer than U chunks, the last maybe half a chunk) follows
  // one chunk at a time.  The first group's weights are asked for before the code table is built: a workgroup lives
  // for little more than one trip to memory, and the table must not stand in front of it.
  const int n_groups = (K >> 7) / U;
  const int n_chunks = (K + 127) >> 7;
  WeightFrag<RT, U> f;
  int j = wave;
  if (j < n_groups) load_weights<RT, U, false>(f, crow, srow, ctile, stile, j * U, true);
  for (int e = t; e < 256; e += blockDim.x)
    lut[e] = make_float2(round_to_bf16(nf4_code_value(e >> 4)), round_to_bf16(nf4_code_value(e & 15)));
  __syncthreads();
  while (j < n_groups) {
    multiply<MT, RT, U, NACC, false>(f, lut, xrow, j * U, true, acc);
    j += nw;
    if (j < n_groups) load_weights<RT, U, false>(f, crow, srow, ctile, stile, j * U, true);
  }
  for (int c = n_groups * U + wave; c < n_chunks; c += nw) {
    const bool valid = c * 128 + 32 * g < K;
    WeightFrag<RT, 1> f1;
    load_weights<RT, 1, true>(f1, crow, srow, ctile, stile, c, valid);
    multiply<MT, RT, 1, NACC, true>(f1, lut, xrow, c, valid, acc);
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int q = 1; q < NACC; ++q) acc[mt][rt][0] += acc[mt][rt][q];
  // acc[mt][rt][0][v] = sum over this wave's chunks of D(W)[n0 + 16 rt + 4 g + v][.] . x[16 mt + i][.]
  if (wave > 0) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int v = 0; v < 4; ++v) red[(((wave - 1) * MT + mt) * RT + rt) * 256 + v * 64 + lane] = acc[mt][rt][0][v];
  }
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int nb = n0 + 16 * rt + 4 * g;  // this lane's four output columns nb .. nb + 3
    float b4[4] = {0.f, 0.f, 0.f, 0.f}, c4[4] = {1.f, 1.f, 1.f, 1.f};
    if (a.bias) {
      const u32x2_t bb = *reinterpret_cast<const u32x2_t*>(a.bias + nb);
      b4[0] = lo_of(bb.x); b4[1] = hi_of(bb.x); b4[2] = lo_of(bb.y); b4[3] = hi_of(bb.y);
    }
    if (a.cscale) {
      const u32x2_t cc = *reinterpret_cast<const u32x2_t*>(a.cscale + nb);
      c4[0] = lo_of(cc.x); c4[1] = hi_of(cc.x); c4[2] = lo_of(cc.y); c4[3] = hi_of(cc.y);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = 16 * mt + i;
      if (m >= a.M) continue;
      float o[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        o[v] = acc[mt][rt][0][v];
        for (int w = 0; w < nw - 1; ++w) o[v] += red[((w * MT + mt) * RT + rt) * 256 + v * 64 + lane];
      }
      if (a.R > 0) {
        // adapter: sum_r bf16(h[m][r] * lscale) * lora_b[n][r], the operands the large-M kernel feeds its MFMA
        float l4[4] = {0.f, 0.f, 0.f, 0.f};
        for (int r0 = 0; r0 < a.R; r0 += 8) {
          const u32x4_t hv = *reinterpret_cast<const u32x4_t*>(a.h + (int64_t)m * a.ldh + r0);
          float hs[8];
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            hs[2 * d] = round_to_bf16(lo_of(hv[d]) * a.lscale);
            hs[2 * d + 1] = round_to_bf16(hi_of(hv[d]) * a.lscale);
          }
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const u32x4_t bv = *reinterpret_cast<const u32x4_t*>(a.lora_b + (int64_t)(nb + v) * a.R + r0);
#pragma unroll
            for (int d = 0; d < 4; ++d) l4[v] += hs[2 * d] * lo_of(bv[d]) + hs[2 * d + 1] * hi_of(bv[d]);
          }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] += l4[v];
      }
      u32x2_t out;
      out.x = pack_pair((o[0] + b4[0]) * c4[0], (o[1] + b4[1]) * c4[1]);
      out.y = pack_pair((o[2] + b4[2]) * c4[2], (o[3] + b4[3]) * c4[3]);
      *reinterpret_cast<u32x2_t*>(a.y + (int64_t)m * a.N + nb) = out;
    }
  }
}

constexpr int kFewTokens = 16;
// The launch shapes below address x, lora_a and the codes of a row tile with 32-bit byte offsets.
constexpr int64_t kFewMaxK = int64_t(1) << 26;
constexpr int kFewHiddenRank = 32;  // most ranks of a member whose hidden product a launch forms itself

// One NF4 code byte's two code points (exact in bf16 and so in fp16) times a block scaler, each one fp32 rounding: the
// conversion rides in the multiply (adding -0 changes no product, signed zeros included).
__device__ __forceinline__ float scaled_lo(uint32_t pair, float s) {
  float r = 0.f;
#if defined(__HIP_DEVICE_COMPILE__)
  asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(s), "s"(-0.0f));
#endif
  return r;
}
__device__ __forceinline__ float scaled_hi(uint32_t pair, float s) {
  float r = 0.f;
#if defined(__HIP_DEVICE_COMPILE__)
  asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(s), "s"(-0.0f));
#endif
  return r;
}

// LDS of a few-token workgroup: the code table, the block scalers of its rows over a segment of the contraction, and per wave
// one stage: 128 columns of x (MQ groups of four tokens), of its row tiles' codes and of its members' lora_a.
template <int RT, int NT, int MQ>
struct FewLayout {
  static constexpr int kCopies = NT > 0 ? 1 : 16;  // of the code table
  static constexpr int kLut = 1024 * kCopies;
  static constexpr int kSegment = 16384 / RT;  // columns; a multiple of 128 times the most waves, so that it does not move the waves' chunks
  static constexpr int kStage = (MQ + RT + 4 * NT) * 1024;
  __host__ __device__ static int scalers(int K) {  // an odd row stride: the rows of a tile on different banks
    const int kb = (K < kSegment ? K : kSegment) >> 6;
    return (RT * 16 * (kb | 1) * 4 + 15) & ~15;
  }
  static int bytes(int K, int waves) { return kLut + scalers(K) + waves * kStage; }
};

// RT tiles of 16 weight rows per workgroup, at most MAXW waves, tokens in MQ groups of four.  PAIR: the even tiles belong to grp.m[0]
// (gate), the odd ones to the same rows of grp.m[1] (up projection, the same width), and act = bf16(bf16(silu(y_0)) * y_1) is
// written as well.
// NA > 0: h = x . lora_a^T is formed here, NA tiles of 16 ranks per member beside the row tiles (the workgroup's own copy: the
// members' first workgroups also write it to m.h_out where that is asked for); otherwise it is read from m.h.
// ONE: the launch has one member, and its arguments sit at fixed places (found through `which` they cost two dependent
// scalar loads before the first request: 0.4 us of a launch of 6 - 8).
template <int RT, int MAXW, int MQ, int NA, bool PAIR, bool ONE>
__global__ __launch_bounds__(64 * MAXW) void nf4_few_kernel(const SmallMGroup grp, uint16_t* __restrict__ act) {
#if defined(__HIP_DEVICE_COMPILE__)  // LDS address-space casts
  static_assert(!PAIR || RT % 2 == 0, "a pair is two row tiles of equal rows");
  constexpr int NT = NA * (PAIR ? 2 : 1);  // rank tiles
  using L = FewLayout<RT, NT, MQ>;
  int which = 0;  // uniform over the workgroup
  if constexpr (!PAIR && !ONE) {
#pragma unroll
    for (int q = 0; q < kGroupMax - 1; ++q)
      if (q < grp.n - 1 && (int)blockIdx.x >= grp.wg_end[q]) which = q + 1;
  }
  extern __shared__ __attribute__((aligned(16))) char few_smem[];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nw = blockDim.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int M = grp.m[which].M, K = grp.m[which].K, KB = K >> 6;
  const int wg = (int)blockIdx.x - (!PAIR && !ONE && which ? grp.wg_end[which - 1] : 0);
  auto member = [&](int rt) -> const SmallMArgs& { return grp.m[PAIR ? rt & 1 : which]; };
  auto first_row = [&](int rt) { return PAIR ? 16 * (wg * (RT / 2) + (rt >> 1)) : 16 * (RT * wg + rt); };  // every row exists
  float* const scal = reinterpret_cast<float*>(few_smem + L::kLut);
  const int scal_bytes = L::scalers(K);
  char* const stage = few_smem + L::kLut + scal_bytes + wave * L::kStage;
  const uint32_t lds_scal = (uint32_t)(uintptr_t)TT_LDS_PTR(scal), lds_stage = (uint32_t)(uintptr_t)TT_LDS_PTR(stage);

  // ---- requests: direct-to-LDS loads, 64 pieces of 16 bytes each.  Four neighbouring lanes ask for 64 contiguous bytes: the
  //      address unit takes them at once, where the lanes of an MFMA operand (neighbours are different rows) cost it four
  //      times as long; that unit was what bounded this kernel.  Piece p of row r of x and lora_a (16 pieces per 128 columns)
  //      goes to slot p ^ r, piece p of row r of the codes (4) to slot p ^ (r / 4) % 4: operand reads then meet no bank twice.
  auto dma16 = [&](uint32_t voff, const void* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds) : "memory", "m0");
  };
  uint32_t x_off[MQ], a_off[NT > 0 ? NA * 4 : 1];
  const int r4 = lane >> 4, p16 = lane & 15, cr = lane >> 2, cp = (lane & 3) ^ ((lane >> 4) & 3);
#pragma unroll
  for (int d = 0; d < MQ; ++d) {
    const int r = 4 * d + r4;
    x_off[d] = (uint32_t)(r < M ? r : M - 1) * (uint32_t)K * 2u + ((p16 ^ r) << 4);  // rows beyond M repeat the last one: never stored
  }
  if constexpr (NT > 0) {
#pragma unroll
    for (int d = 0; d < NA * 4; ++d) {
      const int r = 4 * d + r4;  // ranks beyond R of any member repeat one: zeroed where they would count
      a_off[d] = (uint32_t)r * (uint32_t)K * 2u + ((p16 ^ (r & 15)) << 4);
    }
  }
  const uint32_t c_off = (uint32_t)cr * (uint32_t)(K >> 1) + (cp << 4);
  auto request = [&](int c) {
    const bool half = c * 128 + 64 >= K;  // the last chunk of a K that is an odd multiple of 64: its second half repeats the first
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      dma16(half ? c_off - ((cp & 2) << 4) : c_off, member(rt).codes + (((int64_t)first_row(rt) * K) >> 1) + (int64_t)c * 64,
            lds_stage + (MQ + rt) * 1024);
#pragma unroll
    for (int d = 0; d < MQ; ++d)
      dma16(half ? x_off[d] - (((p16 ^ (4 * d + r4)) & 8) << 4) : x_off[d], reinterpret_cast<const char*>(grp.m[which].x) + (int64_t)c * 256,
            lds_stage + d * 1024);
    if constexpr (NT > 0) {
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        const SmallMArgs& ma = member(a / NA);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const int e = 4 * (a % NA) + d;
          uint32_t off = a_off[e];
          if (4 * e + r4 >= ma.R) off = (p16 ^ ((4 * e + r4) & 15)) << 4;
          if (half) off -= ((p16 ^ ((4 * e + r4) & 15)) & 8) << 4;
          dma16(off, reinterpret_cast<const char*>(ma.lora_a) + (int64_t)c * 256, lds_stage + (MQ + RT + 4 * a) * 1024 + d * 1024);
        }
      }
    }
  };
  constexpr int kBatch = RT + MQ + 4 * NT;
  const int stride = (K < L::kSegment ? KB : L::kSegment >> 6) | 1;
  auto request_scalers = [&](int first, int n) {  // blocks [first, first + n) of every row
    for (int r = wave; r < 16 * RT; r += nw) {
      const float* base = member(PAIR ? r >> 4 : 0).bscal + (int64_t)(first_row(r >> 4) + (r & 15)) * KB + first;
      for (int j = 0; j < n; j += 64)
        if (j + lane < n)
          asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"((uint32_t)(j + lane) * 4u), "s"(base),
                       "s"(lds_scal + (uint32_t)(r * stride + j) * 4u) : "memory", "m0");
    }
  };
  const int n_chunks = (K + 127) >> 7;

  // The first requests leave before the code table is built: a workgroup lives for little more than one trip to memory.
  const int seg_chunks = L::kSegment >> 7;
  request_scalers(0, KB < L::kSegment >> 6 ? KB : L::kSegment >> 6);
  int c = wave;  // the host gives a launch no more waves than there are chunks
  request(c);
  uint32_t* const lut = reinterpret_cast<uint32_t*>(few_smem);
  typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
  for (int e = t; e < 256; e += blockDim.x) {
    const half2_t p = {(_Float16)round_to_bf16(nf4_code_value(e >> 4)), (_Float16)round_to_bf16(nf4_code_value(e & 15))};
    const uint32_t v = __builtin_bit_cast(uint32_t, p);
    if constexpr (L::kCopies == 1) {
      lut[e] = v;
    } else {
#pragma unroll
      for (int j = 0; j < L::kCopies / 4; ++j)
        reinterpret_cast<u32x4_t*>(lut)[e * (L::kCopies / 4) + ((j + e) & (L::kCopies / 4 - 1))] = u32x4_t{v, v, v, v};
    }
  }
  const char* const lut_lane = reinterpret_cast<const char*>(lut) + (L::kCopies > 1 ? (lane & (L::kCopies - 1)) * 4 : 0);
  constexpr int kShift = L::kCopies == 1 ? 2 : 6;  // entry e lies at e << kShift
  auto pair_of = [&](uint32_t codes, int b) {
    const uint32_t off = (8 * b >= kShift ? codes >> (8 * b - kShift) : codes << (kShift - 8 * b)) & (0xffu << kShift);
    return *reinterpret_cast<const uint32_t*>(lut_lane + off);
  };
  constexpr int kChains = 2;  // the same in every instance: a row's bits do not depend on the launch's shape
  f32x4_t acc[RT][kChains], ah[NT > 0 ? NT : 1][kChains];
#pragma unroll
  for (int s = 0; s < kChains; ++s) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[rt][s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < (NT > 0 ? NT : 1); ++a) ah[a][s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  // the scalers are a wave's oldest requests: its first chunk may stay in flight across the barrier
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kBatch) : "memory");

  const int xr = i & (4 * MQ - 1);
  const int x_at = xr * 256, a_at = (MQ + RT) * 1024 + i * 256, c_at = MQ * 1024 + i * 64 + ((g ^ ((i >> 2) & 3)) << 4);
  for (int first = 0;;) {  // segments of the contraction
    const int end = n_chunks < first + seg_chunks ? n_chunks : first + seg_chunks;
    for (; c < end; c += nw) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      // the stage goes to registers and is asked for again
      u32x4_t cd[RT], xb[4], ab[NT > 0 ? NT : 1][4];
      float sc[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        cd[rt] = *reinterpret_cast<const u32x4_t*>(stage + c_at + rt * 1024);
        sc[rt] = scal[(16 * rt + i) * stride + 2 * (c - first) + (g >> 1)];  // beyond K: any value, times zero
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        xb[s] = *reinterpret_cast<const u32x4_t*>(stage + x_at + (((4 * g + s) ^ xr) << 4));
        if constexpr (NT > 0) {
#pragma unroll
          for (int a = 0; a < NT; ++a) ab[a][s] = *reinterpret_cast<const u32x4_t*>(stage + a_at + a * 4096 + (((4 * g + s) ^ i) << 4));
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (c + nw < end) request(c + nw);
      if (c * 128 + 64 >= K && g >= 2) {  // half a chunk: nothing of its second half counts, whatever lies there
#pragma unroll
        for (int s = 0; s < 4; ++s) xb[s] = u32x4_t{0, 0, 0, 0};
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) sc[rt] = 0.f;
        if constexpr (NT > 0) {
#pragma unroll
          for (int a = 0; a < NT; ++a)
#pragma unroll
            for (int s = 0; s < 4; ++s) ab[a][s] = u32x4_t{0, 0, 0, 0};
        }
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bf16x8_t xv = __builtin_bit_cast(bf16x8_t, xb[s]);
        if constexpr (NT > 0) {
#pragma unroll
          for (int a = 0; a < NT; ++a)
            ah[a][s % kChains] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ab[a][s]), xv, ah[a][s % kChains], 0, 0, 0);
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          u32x4_t wf;
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const uint32_t p = pair_of(cd[rt][s], b);
            wf[b] = pack_pair(scaled_lo(p, sc[rt]), scaled_hi(p, sc[rt]));
          }
          acc[rt][s % kChains] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf), xv, acc[rt][s % kChains], 0, 0, 0);
        }
      }
    }
    first += seg_chunks;
    if (first >= n_chunks) break;
    __syncthreads();  // every wave is done with the segment's scalers
    request_scalers(2 * first, KB - 2 * first < (L::kSegment >> 6) ? KB - 2 * first : L::kSegment >> 6);
    if (c < n_chunks) request(c);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  }

  // ---- the waves' partial sums meet in LDS, [tile][lane][v] at the head of each wave's stage, and are added in wave order
  constexpr int kSteps = NA > 0 ? (NA + 1) / 2 : 2;  // MFMA steps of the adapter, 32 ranks each (the ranks of a group add up to at most 64)
  u32x2_t bv[RT][2 * kSteps], hv[PAIR ? 2 : 1][2 * kSteps];  // wave 0: ranks 16 a + 4 g .. + 3 of its rows' lora_b and of its token's h
  if (wave == 0) {
#pragma unroll
    for (int a = 0; a < 2 * kSteps; ++a) {
      const int r = 16 * a + 4 * g;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        bv[rt][a] = u32x2_t{0, 0};
        if (r < member(rt).R) bv[rt][a] = *reinterpret_cast<const u32x2_t*>(member(rt).lora_b + (int64_t)(first_row(rt) + i) * member(rt).R + r);
      }
#pragma unroll
      for (int u = 0; u < (PAIR ? 2 : 1); ++u) {
        hv[u][a] = u32x2_t{0, 0};
        if (NA == 0 && i < M && r < member(u).R) hv[u][a] = *reinterpret_cast<const u32x2_t*>(member(u).h + (int64_t)i * member(u).ldh + r);
      }
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt][0] += acc[rt][1];
  auto leave = [&](int tile, const f32x4_t& v) { *reinterpret_cast<f32x4_t*>(stage + tile * 1024 + lane * 16) = v; };
  if (wave > 0) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) leave(rt, acc[rt][0]);
  }
  if constexpr (NT > 0) {
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      ah[a][0] += ah[a][1];
      if (wave > 0) leave(RT + a, ah[a][0]);
    }
    __syncthreads();
    if (wave == 0) {  // h, rounded to bf16: rank 16 (a % NA) + 4 g + v of token i
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        for (int w = 1; w < nw; ++w) ah[a][0] += *reinterpret_cast<const f32x4_t*>(stage + w * L::kStage + (RT + a) * 1024 + lane * 16);
        const SmallMArgs& ma = member(a / NA);
        const int r = 16 * (a % NA) + 4 * g;
        if (r < ma.R) hv[a / NA][a % NA] = u32x2_t{pack_pair(ah[a][0][0], ah[a][0][1]), pack_pair(ah[a][0][2], ah[a][0][3])};
        if (ma.h_out && wg == 0 && i < M && r < ma.R)
          *reinterpret_cast<u32x2_t*>(ma.h_out + (int64_t)i * ma.ldh + r) = hv[a / NA][a % NA];
      }
    }
  }
  if (wave == 0) {
    // adapter: sum_r bf16(h[m][r] * lscale) * lora_b[n][r], the operands the large-M kernel feeds its MFMA
    auto scaled = [&](uint32_t d, float ls) { return pack_pair(lo_of(d) * ls, hi_of(d) * ls); };
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int u = PAIR ? rt & 1 : 0;
      const float ls = member(rt).lscale;
#pragma unroll
      for (int q = 0; q < kSteps; ++q) {
        if (32 * q >= member(rt).R) break;
        const u32x4_t b = {bv[rt][2 * q].x, bv[rt][2 * q].y, bv[rt][2 * q + 1].x, bv[rt][2 * q + 1].y};
        const u32x4_t h = {scaled(hv[u][2 * q].x, ls), scaled(hv[u][2 * q].y, ls), scaled(hv[u][2 * q + 1].x, ls), scaled(hv[u][2 * q + 1].y, ls)};
        acc[rt][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, h), acc[rt][0], 0, 0, 0);
      }
      leave(rt, acc[rt][0]);
    }
  }
  __syncthreads();
  // every thread finishes one output (PAIR: one of each member) at a time: one wave alone took 1.3 us over sixteen waves' sums
  const char* const parts = few_smem + L::kLut + scal_bytes;
  for (int e = t; e < 256 * (PAIR ? RT / 2 : RT); e += blockDim.x) {
    const int tile = e >> 8, token = (e >> 2) & 15, row = 4 * ((e >> 6) & 3) + (e & 3);
    if (token >= M) continue;
    uint32_t out[PAIR ? 2 : 1];
#pragma unroll
    for (int u = 0; u < (PAIR ? 2 : 1); ++u) {
      const int rt = PAIR ? 2 * tile + u : tile;
      const SmallMArgs& a = member(u);
      const char* p = parts + rt * 1024 + (e & 255) * 4;
      const int n = first_row(rt) + row;
      float o = *reinterpret_cast<const float*>(p);
      if (nw == MAXW) {
#pragma unroll
        for (int w = 1; w < MAXW; ++w) o += *reinterpret_cast<const float*>(p + w * L::kStage);
      } else {
        for (int w = 1; w < nw; ++w) o += *reinterpret_cast<const float*>(p + w * L::kStage);
      }
      if (a.bias) o += bf16_bits_to_f32(a.bias[n]);
      if (a.cscale) o *= bf16_bits_to_f32(a.cscale[n]);
      out[u] = pack_pair(o, 0.f);
      a.y[(int64_t)token * a.N + n] = (uint16_t)out[u];
      if (PAIR && u == 1) act[(int64_t)token * a.N + n] = (uint16_t)swiglu_gate_pair(out[0], out[PAIR ? 1 : 0]);
    }
  }
#endif
}

// Launch shape at most 16 tokens.  The waves fix the order in which a row's products are summed and depend on the
// layer alone, so that a row gets the same bits alone, in a batch of up to 16 tokens and inside a group; row tiles do not
// enter the sums.  Measured over 27 layers of 256 - 28672 rows and 1024 - 28672 columns (us, weights from HBM, launch gap included):
//  * eight waves (4096 x 4096 at 1 / 13 tokens, h formed inside: four 8.7 / 9.3, eight 6.7 / 7.9, sixteen 7.6 / 8.8; 2048 x 8192 at 13: 14.6 /
//    11.1 / 12.3), four where the layer has workgroups to spare and a short contraction (gate / up pair of 14336 x 4096, eight and
//    four: 21.8 and 20.6);
//  * two row tiles, which share the reads of x and lora_a, from 8192 rows on (8192 x 2048 at 13 tokens: one 7.9, two 7.0; 14336 x 4096 at one
//    token with its h: 17.8 and 14.9), but one where four waves at a few tokens read h instead (the same layer 13.9, two 16.1).
struct FewConfig {
  int rt, waves;
  bool operator==(const FewConfig& o) const { return rt == o.rt && waves == o.waves; }
};
int few_waves(int64_t N, int64_t K) { return N > 12288 && K < 8192 ? 4 : 8; }
FewConfig few_config(int64_t M, int64_t N, int64_t K, bool hidden) {
  const int waves = few_waves(N, K);
  return {N >= 8192 && (hidden || waves == 8 || M > 4) ? 2 : 1, waves};
}
FewConfig few_pair_config(int64_t N, int64_t K, bool hidden) {
  const int waves = few_waves(N, K);
  return {hidden && waves == 4 ? 4 : 2, waves};
}
// Whether a launch of these workgroups forms its members' h = x . lora_a^T itself, instead of a launch or two ahead of it (4 - 6.5 us,
// and as many launches for the host).  Every workgroup then reads its members' lora_a, rank_tiles tiles of 16 ranks: at 128 MB
// for the launch still the better way (4096 x 14336: one token 15.6 against 20.2 us, 13 tokens 20.4 against 22.0; at 235 MB, 8192 x
// 28672, no longer), and several tiles only where the LDS they take (`bytes` a workgroup) leaves room for every workgroup at once
// (gate / up pair of 8192 x 2048, 512 workgroups in two rounds: 15.1 against 12.1; in one round, 2816 x 1024: 6.8 against 8.7).
bool few_hidden(int64_t workgroups, int rank_tiles, int64_t K, int bytes) {
  if (rank_tiles > 1 && workgroups > 256 * (160 * 1024 / bytes)) return false;
  return workgroups * rank_tiles * 32 * K <= int64_t(128) << 20;
}
int few_bytes(int rt, int rank_tiles, int64_t M, int64_t K, int waves) {
  const int cols = 16384 / rt, kb = (int)(K < cols ? K : cols) >> 6, n_chunks = (int)((K + 127) >> 7);
  return 1024 + 64 * rt * (kb | 1) + (n_chunks < waves ? n_chunks : waves) * ((M <= 4 ? 1 : 4) + rt + 4 * rank_tiles) * 1024;
}

template <int RT, int MAXW, int MQ, int NA, bool PAIR, bool ONE>
int launch_few(const SmallMGroup& g, unsigned wgs, uint16_t* act, hipStream_t s) {
  constexpr int NT = NA * (PAIR ? 2 : 1);
  using L = FewLayout<RT, NT, MQ>;
  const int K = g.m[0].K, n_chunks = (K + 127) >> 7, waves = n_chunks < MAXW ? n_chunks : MAXW;
  static bool attr_set[64] = {};  // the LDS limit is a per-device attribute of the function
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (dev < 0 || !attr_set[dev]) {
    const int most = L::bytes(L::kSegment, MAXW);
    static_assert(FewLayout<RT, NT, MQ>::kLut + 16 * RT * (16384 / RT / 64 + 1) * 4 + MAXW * FewLayout<RT, NT, MQ>::kStage <= 160 * 1024,
                  "the LDS of a CU");
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&nf4_few_kernel<RT, MAXW, MQ, NA, PAIR, ONE>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, most);
    if (e != hipSuccess) return fail(TTAMD_ELAUNCH, "nf4_few: cannot reserve %d bytes of LDS: %s", most, hipGetErrorString(e));
    if (dev >= 0) attr_set[dev] = true;
  }
  nf4_few_kernel<RT, MAXW, MQ, NA, PAIR, ONE><<<dim3(wgs), dim3(64 * waves), L::bytes(K, waves), s>>>(g, act);
  return check_launch("nf4_few");
}

template <int RT, int MAXW, int MQ, int NA>
int launch_few_members(SmallMGroup& g, hipStream_t s) {
  int wgs = 0;
  for (int i = 0; i < g.n; ++i) {
    wgs += g.m[i].N / (16 * RT);
    g.wg_end[i] = wgs;
  }
  return g.n == 1 ? launch_few<RT, MAXW, MQ, NA, false, true>(g, wgs, nullptr, s) : launch_few<RT, MAXW, MQ, NA, false, false>(g, wgs, nullptr, s);
}

// rank_tiles: of a member, where the launch forms h; 0 where it reads it
template <int MQ, int NA>
int dispatch_few_members(SmallMGroup& g, const FewConfig& c, hipStream_t s) {
  if (c.rt == 1) {
    if constexpr (MQ == 1 && NA == 0) {
      if (c.waves == 4) return launch_few_members<1, 4, MQ, NA>(g, s);
    }
    return launch_few_members<1, 8, MQ, NA>(g, s);
  }
  return c.waves == 8 ? launch_few_members<2, 8, MQ, NA>(g, s) : launch_few_members<2, 4, MQ, NA>(g, s);
}
int dispatch_few(SmallMGroup& g, const FewConfig& c, int rank_tiles, hipStream_t s) {
  const bool one = g.m[0].M <= 4;  // group of four tokens
  switch (rank_tiles) {
    case 0: return one ? dispatch_few_members<1, 0>(g, c, s) : dispatch_few_members<4, 0>(g, c, s);
    case 1: return one ? dispatch_few_members<1, 1>(g, c, s) : dispatch_few_members<4, 1>(g, c, s);
    default: return one ? dispatch_few_members<1, 2>(g, c, s) : dispatch_few_members<4, 2>(g, c, s);
  }
}
int dispatch_few_pair(const SmallMGroup& g, const FewConfig& c, bool hidden, uint16_t* act, hipStream_t s) {
  const unsigned wgs = g.m[0].N / (8 * c.rt);
  const bool one = g.m[0].M <= 4;
  if (hidden) {
    if (c.rt == 4) return launch_few<4, 4, 1, 1, true, false>(g, wgs, act, s);  // few_pair_hidden: at most four tokens
    return one ? launch_few<2, 8, 1, 1, true, false>(g, wgs, act, s) : launch_few<2, 8, 4, 1, true, false>(g, wgs, act, s);
  }
  if (c.waves == 4) return one ? launch_few<2, 4, 1, 0, true, false>(g, wgs, act, s) : launch_few<2, 4, 4, 0, true, false>(g, wgs, act, s);
  return one ? launch_few<2, 8, 1, 0, true, false>(g, wgs, act, s) : launch_few<2, 8, 4, 0, true, false>(g, wgs, act, s);
}

// Shape of a launch of 17 - 64 tokens: token tiles, row tiles per workgroup, chunks in flight per wave, most waves.  It fixes
// the order in which a row's products are summed, so a layer gets the same bits alone and inside a group.
struct SmallMConfig {
  int mt, rt, u, max_waves;
  bool operator==(const SmallMConfig& o) const { return mt == o.mt && rt == o.rt && u == o.u && max_waves == o.max_waves; }
};
// Measured on MI355X over the projections of an 8B model (kernel time, M = 32 / 64): 4096 x 4096 13 / 20 us, 14336 x 4096
// 26 / 43 us, 4096 x 14336 37 / 64 us.  Wide layers share an x fragment between two row tiles (x comes from L2 once per
// workgroup); long contractions of four token tiles get sixteen waves, the others four.
SmallMConfig small_m_config(int64_t M, int64_t N, int64_t K) {
  const bool wide = N >= 8192, deep = K >= 8192;
  if (M <= 32) return wide ? SmallMConfig{2, 2, 4, 4} : SmallMConfig{2, 1, 4, 4};
  return wide ? SmallMConfig{4, 2, 2, 4} : SmallMConfig{4, 1, 4, deep ? 16 : 4};
}

template <int MT, int RT, int U, int MAXW>
int launch_small_m(SmallMGroup& g, hipStream_t s) {
  static_assert(MAXW <= kSmMaxWaves, "the partial sums are laid out for at most kSmMaxWaves waves");
  const int K = g.m[0].K;
  int nw = ((K >> 7) + U - 1) / U;  // one group of U chunks per wave when K is short enough
  nw = nw > 1 ? nw : 1;
  nw = nw < MAXW ? nw : MAXW;
  // the partial sums of waves 1 .. nw - 1 must fit the 64 KB of LDS a workgroup gets without asking for more
  const int per_wave = MT * RT * 4 * 64 * (int)sizeof(float);
  const int fit = 1 + (63 * 1024) / per_wave;
  nw = nw < fit ? nw : fit;
  int wgs = 0;
  for (int i = 0; i < g.n; ++i) {
    wgs += g.m[i].N / (16 * RT);
    g.wg_end[i] = wgs;
  }
  const dim3 grid((unsigned)wgs), block(64 * nw);
  nf4_small_m_kernel<MT, RT, U, MAXW><<<grid, block, (size_t)(nw - 1) * per_wave, s>>>(g);
  return check_launch("nf4_small_m");
}

int dispatch_small_m(SmallMGroup& g, const SmallMConfig& c, hipStream_t s) {
  if (c.mt == 2) return c.rt == 2 ? launch_small_m<2, 2, 4, 4>(g, s) : launch_small_m<2, 1, 4, 4>(g, s);
  if (c.rt == 2) return launch_small_m<4, 2, 2, 4>(g, s);
  return c.max_waves > 4 ? launch_small_m<4, 1, 4, 16>(g, s) : launch_small_m<4, 1, 4, 4>(g, s);
}

}  // namespace

// Largest token count the small-M kernel takes; above it the tiled kernel runs.
int small_m_limit() { return 64; }

// Whether a forward of M tokens on an [N, K] weight goes to this kernel.  sliced_ok: the caller brought the workspace
// that lets the tiled kernel cut its contraction into slices.  Without it the tiled kernel fills 16 - 56 workgroups at
// these sizes and this kernel wins up to 64 tokens.  With it (measured, us, few-token / sliced at 24, 32, 40, 64 tokens):
// 4096 x 4096 13 / 17, 14 / 18, 20 / 19, 25 / 22; 14336 x 4096 29 / 23, 31 / 24, 40 / 25, 50 / 27; 4096 x 14336 33 / 24,
// 37 / 25, 50 / 26, 66 / 28: every workgroup of this kernel reads all of x, which at 64 tokens is seven times the
// packed weight, so from 17 tokens on the large weights and from 33 on all of them are better off in slices.
bool small_m_applies(int64_t M, int64_t N, int64_t K, bool sliced_ok) {
  if (M > small_m_limit()) return false;
  if (M <= 16 || !sliced_ok) return true;
  return M <= 32 && N * K <= (int64_t(1) << 25);
}

// Entries used by the C-ABI wrappers (arguments already validated there: N % 64 == 0, K % 64 == 0, R % 8 == 0, pointers
// aligned).  `bscal` is the natural [N, K/64] scaler layout; the rows of `h` are ldh elements apart.
int run_small_m(const void* x, const uint8_t* codes, const void* bscal, const void* h, int ldh, const void* lora_b, int R,
                float lscale, const void* bias, const void* cscale, void* y, int64_t M, int64_t N, int64_t K, hipStream_t s) {
  TT_REQUIRE(M > 0 && M <= small_m_limit(), "nf4_small_m: M (%lld) out of range", (long long)M);
  TT_REQUIRE(N / 16 < (int64_t(1) << 31) && N * K < (int64_t(1) << 40), "nf4_small_m: weight too large");
  SmallMGroup g = {};
  g.n = 1;
  SmallMArgs& a = g.m[0];
  a.x = reinterpret_cast<const uint16_t*>(x);
  a.codes = codes;
  a.bscal = reinterpret_cast<const float*>(bscal);
  a.h = reinterpret_cast<const uint16_t*>(h);
  a.lora_b = reinterpret_cast<const uint16_t*>(lora_b);
  a.bias = reinterpret_cast<const uint16_t*>(bias);
  a.cscale = reinterpret_cast<const uint16_t*>(cscale);
  a.y = reinterpret_cast<uint16_t*>(y);
  a.M = (int)M; a.N = (int)N; a.K = (int)K; a.R = R; a.ldh = ldh;
  a.lscale = lscale;
  if (M <= kFewTokens && K < kFewMaxK) return dispatch_few(g, few_config(M, N, K, false), 0, s);
  return dispatch_small_m(g, small_m_config(M, N, K), s);
}

namespace {
int small_m_args(SmallMArgs (&all)[kGroupMax], const void* x, const GroupGemm& gg, const void* h_cat) {
  TT_REQUIRE(gg.M > 0 && gg.M <= small_m_limit(), "nf4_small_m: M (%lld) out of range", (long long)gg.M);
  for (int j = 0; j < gg.n; ++j) {
    TT_REQUIRE(gg.N[j] / 16 < (int64_t(1) << 27) && gg.N[j] * gg.K < (int64_t(1) << 40), "nf4_small_m: weight too large");
    SmallMArgs& a = all[j];
    a.x = reinterpret_cast<const uint16_t*>(x);
    a.codes = gg.codes[j];
    a.bscal = gg.bscal[j];
    a.h = h_cat ? reinterpret_cast<const uint16_t*>(h_cat) + gg.r_off[j] : nullptr;
    a.lora_b = gg.lora_b[j];
    a.bias = gg.bias[j];
    a.y = gg.y[j];
    a.M = (int)gg.M; a.N = (int)gg.N[j]; a.K = (int)gg.K; a.R = gg.rank[j]; a.ldh = gg.r_off[gg.n];
    a.lscale = gg.scale[j];
  }
  return TTAMD_OK;
}
// members [i, j) share a launch
template <typename Same>
int run_of(const GroupGemm& gg, int i, Same same) {
  int j = i + 1;
  while (j < gg.n && same(i, j)) ++j;
  return j;
}
bool same_few(const GroupGemm& gg, int i, int j, bool hidden) {
  return few_config(gg.M, gg.N[j], gg.K, hidden) == few_config(gg.M, gg.N[i], gg.K, hidden);
}
int rank_tiles_of(const GroupGemm& gg, int i, int j) {
  int most = 0;
  for (int q = i; q < j; ++q) most = gg.rank[q] > most ? gg.rank[q] : most;
  return (most + 15) / 16;
}
}  // namespace

// The members of a group (same x, M, K) in as few launches as their launch shapes allow: consecutive members with
// the same shape share one.  act != nullptr (two members of equal width): *act_done says whether the launch wrote
// act = silu(y_0) * y_1 too.
int run_small_m_group(const void* x, const GroupGemm& gg, const void* h_cat, void* act, bool* act_done, hipStream_t s) {
  SmallMArgs all[kGroupMax] = {};
  if (int rc = small_m_args(all, x, gg, h_cat)) return rc;
  const bool few = gg.M <= kFewTokens && gg.K < kFewMaxK;
  if (act && few && gg.n == 2 && gg.N[0] == gg.N[1]) {
    SmallMGroup g = {};
    g.m[0] = all[0];
    g.m[1] = all[1];
    g.n = 2;
    *act_done = true;
    return dispatch_few_pair(g, few_pair_config(gg.N[0], gg.K, false), false, reinterpret_cast<uint16_t*>(act), s);
  }
  for (int i = 0; i < gg.n;) {
    SmallMGroup g = {};
    const int j = run_of(gg, i, [&](int p, int q) {
      return few ? same_few(gg, p, q, false) : small_m_config(gg.M, gg.N[q], gg.K) == small_m_config(gg.M, gg.N[p], gg.K);
    });
    for (int q = i; q < j; ++q) g.m[q - i] = all[q];
    g.n = j - i;
    if (int rc = few ? dispatch_few(g, few_config(gg.M, gg.N[i], gg.K, false), 0, s) : dispatch_small_m(g, small_m_config(gg.M, gg.N[i], gg.K), s)) return rc;
    i = j;
  }
  return TTAMD_OK;
}

bool few_forms_hidden(const GroupGemm& gg, bool gated) {
  if (gg.M > kFewTokens || gg.K >= kFewMaxK) return false;
  for (int i = 0; i < gg.n; ++i)
    if (gg.rank[i] < 8 || gg.rank[i] > kFewHiddenRank) return false;
  if (gated) {
    const FewConfig c = few_pair_config(gg.N[0], gg.K, true);
    return rank_tiles_of(gg, 0, 2) == 1 && (c.rt == 2 || gg.M <= 4) && few_hidden(gg.N[0] / (8 * c.rt), 2, gg.K, few_bytes(c.rt, 2, gg.M, gg.K, c.waves));
  }
  for (int i = 0; i < gg.n;) {
    const int j = run_of(gg, i, [&](int p, int q) { return same_few(gg, p, q, true); });
    int64_t wgs = 0;
    for (int q = i; q < j; ++q) wgs += gg.N[q] / (16 * few_config(gg.M, gg.N[q], gg.K, true).rt);
    const FewConfig c = few_config(gg.M, gg.N[i], gg.K, true);
    const int tiles = rank_tiles_of(gg, i, j);
    if (!few_hidden(wgs, tiles, gg.K, few_bytes(c.rt, tiles, gg.M, gg.K, c.waves))) return false;
    i = j;
  }
  return true;
}

int run_few_with_hidden(const void* x, const GroupGemm& gg, const uint16_t* const* lora_a, void* h_cat, void* act, hipStream_t s) {
  SmallMArgs all[kGroupMax] = {};
  if (int rc = small_m_args(all, x, gg, nullptr)) return rc;
  for (int q = 0; q < gg.n; ++q) {
    all[q].lora_a = lora_a[q];
    all[q].h_out = h_cat ? reinterpret_cast<uint16_t*>(h_cat) + gg.r_off[q] : nullptr;
  }
  SmallMGroup g = {};
  if (act) {
    g.m[0] = all[0];
    g.m[1] = all[1];
    g.n = 2;
    return dispatch_few_pair(g, few_pair_config(gg.N[0], gg.K, true), true, reinterpret_cast<uint16_t*>(act), s);
  }
  for (int i = 0; i < gg.n;) {
    const int j = run_of(gg, i, [&](int p, int q) { return same_few(gg, p, q, true); });
    for (int q = i; q < j; ++q) g.m[q - i] = all[q];
    g.n = j - i;
    if (int rc = dispatch_few(g, few_config(gg.M, gg.N[i], gg.K, true), rank_tiles_of(gg, i, j), s)) return rc;
    i = j;
  }
  return TTAMD_OK;
}

}  // namespace ttamd
