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
//    us, weights from HBM, hidden product included, before -> now at 1 / 13 tokens: 4096 x 4096 12.5 / 14.2 -> 7.9 / 8.4, 14336 x 4096 21.3 /
//    25.7 -> 17.0 / 19.7, 4096 x 14336 22.1 / 30.8 -> 19.3 / 23.3, 2048 x 2048 9.1 / 11.1 -> 5.6 / 6.1, gate / up pair of 14336 x 4096 38.0 / 43.1 ->
//    31.0 / 31.5.  A read of the same bytes in the same row pieces takes 3.1, 6.3, 6.6 and (the pair) 10.3: the pair is bound by
//    the expansion (VALU 10.9 us, LDS 11.7 of 22 us busy without the hidden product).
//  * nf4_small_m_kernel (17 - 64 tokens): groups of U chunks per wave, two or four token tiles.
#include "common.h"
#include "group.h"
#include "nf4_math.h"
#include "swiglu_math.h"

#include <type_traits>

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
  int splits, chunks_per_split;  // where the launch forms h: how its sums run (hidden_order)
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

constexpr int kFewTokens = TTAMD_FEW_TOKENS;
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

// How h = x . lora_a^T of at most 16 tokens is summed, wherever it is formed: the order of the adapters' own launch
// (lora_skinny.hip), which is the same for every such token count, for a member alone and in a group.
//   K <= kNtFewK (splits == 0): 64-wide chunks go round sixteen waves, two chains each (the halves of every chunk); the chains of
//     a wave, then the waves in order.
//   beyond: splits of chunks_per_split chunks, dealt to four waves in turn, one chain each; the waves of a split in order,
//     then the splits.
// In a chunk lane group g holds columns 16 g .. + 15, the first eight for one MFMA, the others for the next.
// A launch that forms h itself meets that order by one of three forms:
//   kWaves (splits == 0): the 128-wide chunk that a wave has staged for its weight rows is a chunk of two of the sixteen waves.
//   kPaired (sixteen parts of a row's sum, eight chunks per split): the two parts of a wave are two 128-wide chunks apart, which
//     makes them the two chunks of two chains.
//   kGather (the others): the chunks of a chain, a and a + 4, are staged side by side, x a second time with them; a wave forms
//     whole splits.
enum HiddenForm { kReads, kWaves, kPaired, kGather };

// LDS of a few-token workgroup: the code table, the block scalers of its rows over a segment of the contraction, the splits'
// sums of h, and per wave one stage: 128 columns of x (MQ groups of four tokens), of its row tiles' codes, and of its
// members' lora_a (kGather: and of x again).  At the end a stage holds the wave's partial sums.
// Sixteen copies of the code table where h is read (us behind one another in a graph, sixteen and one: 14336 x 4096 at one token
// 13.3 and 14.2, 9728 x 3584 10.2 and 11.2, 28672 x 8192 36.6 and 38.3; 4096 x 4096 level; their fill costs small layers 2 - 5 %, 2048 x
// 2048 4.5 and 4.3, and their LDS a workgroup per CU at 28672 x 8192 from 8 tokens on, 45.7 and 41.3), one where it is formed: LDS
// has the operands of h to hold.
constexpr int few_lut_bytes(int nt) { return nt > 0 ? 1024 : 16 * 1024; }
// Columns of a segment: whole rounds of the waves' chunks and splits, so that it does not move either.
constexpr int few_segment(int rt, int nt, int mq, int form) {
  return nt == 2 && mq == 4 ? 4096 : form == kPaired && mq == 4 ? 8192 : 16384 / rt;
}
constexpr int few_stage_bytes(int rt, int sets, int nt, int mq, int form) {
  const int staged = mq + rt + (form == kGather ? mq : 0) + 4 * nt, left = sets * rt;
  return (staged > left ? staged : left) * 1024;
}
constexpr int few_scaler_bytes(int rt, int nt, int mq, int form, int K) {  // an odd row stride: the rows of a tile on different banks
  const int segment = few_segment(rt, nt, mq, form), kb = (K < segment ? K : segment) >> 6;
  return (rt * 16 * (kb | 1) * 4 + 15) & ~15;
}
// fp32 [split][sums of a split][rank tile][4 ranks][token][4]; kPaired: of its first two chains, its third, its fourth
constexpr int few_split_sums(int form) { return form == kPaired ? 3 : form == kGather ? 1 : 0; }
constexpr int few_split_bytes(int rt, int nt, int mq, int form, int splits) {
  const int most = few_segment(rt, nt, mq, form) / 512;
  return (splits < most ? splits : most) * few_split_sums(form) * nt * 64 * 4 * mq;
}
constexpr int few_bytes(int rt, int sets, int nt, int mq, int form, int K, int splits, int waves) {
  return few_lut_bytes(nt) + few_scaler_bytes(rt, nt, mq, form, K) + few_split_bytes(rt, nt, mq, form, splits) +
         waves * few_stage_bytes(rt, sets, nt, mq, form);
}

// RT tiles of 16 weight rows per workgroup, at most MAXW waves, tokens in MQ groups of four.  PAIR: the even tiles belong to grp.m[0]
// (gate), the odd ones to the same rows of grp.m[1] (up projection, the same width), and act = bf16(bf16(silu(y_0)) * y_1) is
// written as well.
// SETS: a row's chunks are summed in MAXW SETS parts of four chains each (part c % (MAXW SETS) takes chunk c), added in order; a
// wave has the parts wave and wave + 8, kPaired: 4 (wave / 2) + wave % 2 and the one two further on.
// FORM != kReads: h = x . lora_a^T is formed here, NA tiles of 16 ranks per member beside the row tiles (the workgroup's own
// copy: the members' first workgroups also write it to m.h_out where that is asked for); otherwise it is read from m.h.
// ONE: the launch has one member, and its arguments sit at fixed places (found through `which` they cost two dependent
// scalar loads before the first request: 0.4 us of a launch of 6 - 8).
// Registers: two workgroups per CU, but one of eight waves where LDS has no room for a second.
template <int RT, int MAXW, int SETS, int MQ, int NA, int FORM, bool PAIR, bool ONE>
__global__ __launch_bounds__(64 * MAXW, MAXW == 8 && NA * (PAIR ? 2 : 1) <= 1 && (FORM < kPaired || MQ == 1) ? 4 : 2) void nf4_few_kernel(const SmallMGroup grp, uint16_t* __restrict__ act) {
#if defined(__HIP_DEVICE_COMPILE__)  // LDS address-space casts
  static_assert(!PAIR || RT % 2 == 0, "a pair is two row tiles of equal rows");
  static_assert(MAXW == 8 || (MAXW == 4 && SETS == 1), "the parts of a row's sum");
  constexpr int NT = NA * (PAIR ? 2 : 1), kNA = NA > 0 ? NA : 1;  // rank tiles, of a member
  constexpr bool GATHER = FORM == kGather, PAIRED = FORM == kPaired, SPLITS = GATHER || PAIRED;
  static_assert((NA > 0) == (FORM != kReads) && (!PAIRED || (MAXW == 8 && SETS == 2)), "the forms");
  constexpr int kStage = few_stage_bytes(RT, SETS, NT, MQ, FORM), kSegment = few_segment(RT, NT, MQ, FORM);
  constexpr int kX2 = (MQ + RT) * 1024, kA = kX2 + (GATHER ? MQ * 1024 : 0);  // of a stage: x again, lora_a
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
  float* const scal = reinterpret_cast<float*>(few_smem + few_lut_bytes(NT));
  const int n_splits = SPLITS ? grp.splits : 0, per_split = grp.chunks_per_split;
  char* const split_sums = few_smem + few_lut_bytes(NT) + few_scaler_bytes(RT, NT, MQ, FORM, K);
  char* const stages = split_sums + few_split_bytes(RT, NT, MQ, FORM, n_splits);
  char* const stage = stages + wave * kStage;
  const uint32_t lds_scal = (uint32_t)(uintptr_t)TT_LDS_PTR(scal), lds_stage = (uint32_t)(uintptr_t)TT_LDS_PTR(stage);

  // ---- requests: direct-to-LDS loads, 64 pieces of 16 bytes each.  Four neighbouring lanes ask for 64 contiguous bytes: the
  //      address unit takes them at once, where the lanes of an MFMA operand (neighbours are different rows) cost it four
  //      times as long; that unit was what bounded this kernel.  Piece p of row r of x and lora_a (16 pieces per 128 columns)
  //      goes to slot p ^ r, piece p of row r of the codes (4) to slot p ^ (r / 4) % 4: operand reads then meet no bank twice.
  auto dma16 = [&](uint32_t voff, const void* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds) : "memory", "m0");
  };
  const int r4 = lane >> 4, cr = lane >> 2, cp = (lane & 3) ^ ((lane >> 4) & 3);
  uint32_t piece[4];  // byte offset of the lane's piece of row 4 d + r4 (and of the rows 16 further on)
  uint32_t x_row[MQ];
#pragma unroll
  for (int d = 0; d < 4; ++d) piece[d] = (uint32_t)((lane & 15) ^ (4 * d + r4)) << 4;
#pragma unroll
  for (int d = 0; d < MQ; ++d) {
    const int r = 4 * d + r4;
    x_row[d] = (uint32_t)(r < M ? r : M - 1) * (uint32_t)K * 2u;  // rows beyond M repeat the last one: never stored
  }
  const uint32_t a_lane = (uint32_t)r4 * (uint32_t)K * 2u;
  auto request_x = [&](int64_t col_bytes, int to, auto at) {
#pragma unroll
    for (int d = 0; d < MQ; ++d) dma16(x_row[d] + at(piece[d]), reinterpret_cast<const char*>(grp.m[which].x) + col_bytes, lds_stage + to + d * 1024);
  };
  auto request_a = [&](int64_t col_bytes, auto at) {
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      const SmallMArgs& ma = member(a / kNA);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const int row = 16 * (a % kNA) + 4 * d;  // R % 8 == 0: four rows exist or none; beyond R the first ones again, which do not count
        dma16(a_lane + at(piece[d]), reinterpret_cast<const char*>(ma.lora_a) + (row < ma.R ? (int64_t)row * K * 2 : 0) + col_bytes,
              lds_stage + kA + a * 4096 + d * 1024);
      }
    }
  };
  const uint32_t c_off = (uint32_t)cr * (uint32_t)(K >> 1) + (cp << 4);
  auto half_of = [&](int c) { return c * 128 + 64 >= K; };  // the last chunk of a K that is an odd multiple of 64: its second half repeats the first
  auto request_codes = [&](int c) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      dma16(half_of(c) ? c_off - ((cp & 2) << 4) : c_off, member(rt).codes + (((int64_t)first_row(rt) * K) >> 1) + (int64_t)c * 64,
            lds_stage + (MQ + rt) * 1024);
  };
  auto request_operands = [&](int c) {
    const uint32_t mask = half_of(c) ? 0x70u : 0xf0u;
    auto at = [&](uint32_t p) { return p & mask; };
    request_x((int64_t)c * 256, 0, at);
    if constexpr (NT > 0 && !GATHER) request_a((int64_t)c * 256, at);
  };
  auto request = [&](int c) {
    request_codes(c);
    request_operands(c);
  };
  // GATHER: chain w of split sp; its chunks are chunk_of and, where that exists, four further on
  auto chunk_of = [&](int sp, int w) { return sp * per_split + w; };
  auto chunks_end = [&](int sp) { return (sp + 1) * per_split < KB ? (sp + 1) * per_split : KB; };
  auto request_chain = [&](int sp, int w) {
    const uint32_t second = chunk_of(sp, w) + 4 < chunks_end(sp) ? 512u : 0u;  // otherwise the second repeats the first
    auto at = [&](uint32_t p) { return (p & 0x70u) | ((p << 2) & second); };
    request_x((int64_t)chunk_of(sp, w) * 128, kX2, at);
    request_a((int64_t)chunk_of(sp, w) * 128, at);
  };
  const int stride = (K < kSegment ? KB : kSegment >> 6) | 1;
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
  constexpr int seg_chunks = kSegment >> 7, seg_splits = kSegment / 512;
  request_scalers(0, KB < kSegment >> 6 ? KB : kSegment >> 6);
  const int start = PAIRED ? 4 * (wave >> 1) + (wave & 1) : wave;  // the wave's first chunk of a segment
  request(start);  // the host gives a launch no more waves than there are chunks (kPaired: at least seventeen chunks)
  if constexpr (GATHER) {
    if (wave < n_splits) request_chain(wave, 0);
  }
  uint32_t* const lut = reinterpret_cast<uint32_t*>(few_smem);
  constexpr int kCopies = few_lut_bytes(NT) / 1024;
  typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
  for (int e = t; e < 256; e += blockDim.x) {
    const half2_t p = {(_Float16)round_to_bf16(nf4_code_value(e >> 4)), (_Float16)round_to_bf16(nf4_code_value(e & 15))};
    const uint32_t v = __builtin_bit_cast(uint32_t, p);
    if constexpr (kCopies == 1) {
      lut[e] = v;
    } else {
#pragma unroll
      for (int j = 0; j < kCopies / 4; ++j)
        reinterpret_cast<u32x4_t*>(lut)[e * (kCopies / 4) + ((j + e) & (kCopies / 4 - 1))] = u32x4_t{v, v, v, v};
    }
  }
  const char* const lut_lane = reinterpret_cast<const char*>(lut) + (kCopies > 1 ? (lane & (kCopies - 1)) * 4 : 0);
  constexpr int kShift = kCopies == 1 ? 2 : 6;  // entry e lies at e << kShift
  auto pair_of = [&](uint32_t codes, int b) {
    const uint32_t off = (8 * b >= kShift ? codes >> (8 * b - kShift) : codes << (kShift - 8 * b)) & (0xffu << kShift);
    return *reinterpret_cast<const uint32_t*>(lut_lane + off);
  };
  constexpr int kHSets = SPLITS ? 1 : 8 / MAXW;  // pairs of h's sixteen parts that a wave forms
  // h: kWaves [][set][half of a chunk][chain]; kPaired [][0][chain][0]; kGather [][0][0][0] the split's sum so far
  f32x4_t acc[RT][SETS][4], ah[NT > 0 ? NT : 1][kHSets][2][2];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int u = 0; u < SETS; ++u) acc[rt][u][s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < (NT > 0 ? NT : 1); ++a)
#pragma unroll
      for (int u = 0; u < kHSets; ++u) ah[a][u][s >> 1][s & 1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  // the scalers are a wave's oldest requests: its first chunk (and chain) may stay in flight across the barrier
  if (GATHER && wave >= n_splits)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(RT + MQ) : "memory");
  else
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(RT + MQ + (GATHER ? MQ : 0) + 4 * NT) : "memory");

  constexpr int kTokens = 4 * MQ;
  const int xr = i & (kTokens - 1);
  const int c_at = MQ * 1024 + i * 64 + ((g ^ ((i >> 2) & 3)) << 4);
  // piece p of this lane's token and rank
  auto read_x = [&](int from, int p) { return *reinterpret_cast<const u32x4_t*>(stage + from + xr * 256 + ((p ^ xr) << 4)); };
  auto read_a = [&](int a, int p) { return *reinterpret_cast<const u32x4_t*>(stage + kA + a * 4096 + i * 256 + ((p ^ i) << 4)); };
  auto mfma = [&](const u32x4_t& rows, const u32x4_t& cols, const f32x4_t& sum) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, rows), __builtin_bit_cast(bf16x8_t, cols), sum, 0, 0, 0);
  };
  // what this thread has of h where splits are added, elements t, t + 64 MAXW, .. of [rank tile][4 ranks][token][4]
  constexpr int kHElements = NT * 16 * kTokens, kHOwn = (kHElements + 64 * MAXW - 1) / (64 * MAXW);
  float h_sum[kHOwn > 0 ? kHOwn : 1];
#pragma unroll
  for (int j = 0; j < (kHOwn > 0 ? kHOwn : 1); ++j) h_sum[j] = 0.f;

  for (int first = 0;;) {  // segments of the contraction
    const int end = n_chunks < first + seg_chunks ? n_chunks : first + seg_chunks;
    const int first_split = first / seg_chunks * seg_splits, end_split = n_splits < first_split + seg_splits ? n_splits : first_split + seg_splits;
    // One chunk of the weight rows and (GATHER) one chain of h.  set: the part of the sums that they belong to.
    int c = first + start, sp = first_split + wave, w = 0;
    auto step = [&](auto which_set) {
      constexpr int set = decltype(which_set)::value;
      const int next = PAIRED ? (set == 0 ? c + 2 : c + 14) : c + nw;
      const bool has = c < end;
      const int chunk = GATHER && sp < end_split ? chunk_of(sp, w) : 0, stop = GATHER && sp < end_split ? chunks_end(sp) : 0;
      const bool chain = GATHER && chunk < stop;
      const bool half = half_of(c);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      // the stage goes to registers and is asked for again
      u32x4_t cd[RT], xb[4], xh[4], ab[NT > 0 ? NT : 1][4];
      float sc[RT];
      const bool forms = NT > 0 && (GATHER ? chain : has);
      auto multiply_h = [&]() {
        if (!forms) return;
#pragma unroll
        for (int a = 0; a < NT; ++a) {
          if constexpr (GATHER) {
            f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
            sum = mfma(ab[a][1], xh[1], mfma(ab[a][0], xh[0], sum));
            if (chunk + 4 < stop) sum = mfma(ab[a][3], xh[3], mfma(ab[a][2], xh[2], sum));
            ah[a][0][0][0] = w == 0 ? sum : ah[a][0][0][0] + sum;
          } else if constexpr (PAIRED) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              if (set == 0) ah[a][0][b][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
              if (b == 0 || !half) ah[a][0][b][0] = mfma(ab[a][2 * b + 1], xh[2 * b + 1], mfma(ab[a][2 * b], xh[2 * b], ah[a][0][b][0]));
            }
          } else {
            constexpr int hs = set % kHSets;
#pragma unroll
            for (int s = 0; s < 4; ++s)
              if (s < 2 || !half) ah[a][hs][s >> 1][s & 1] = mfma(ab[a][s], xh[s], ah[a][hs][s >> 1][s & 1]);
          }
        }
      };
      auto read_h = [&]() {
        if (!forms) return;
#pragma unroll
        for (int s = 0; s < 4; ++s) {  // half s / 2 of the 128 columns, MFMA s % 2 of it
          const int p = 8 * (s >> 1) + 2 * g + (s & 1);
          xh[s] = read_x(GATHER ? kX2 : 0, p);
#pragma unroll
          for (int a = 0; a < NT; ++a) ab[a][s] = read_a(a, p);
        }
      };
      constexpr bool kHFirst = NT > 0 && RT > 1;  // all operands at once do not fit the registers of two workgroups per CU
      if constexpr (kHFirst) {
        read_h();
        multiply_h();
        asm volatile("" ::: "memory");
      }
      if (has) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          cd[rt] = *reinterpret_cast<const u32x4_t*>(stage + c_at + rt * 1024);
          sc[rt] = scal[(16 * rt + i) * stride + 2 * (c - first) + (g >> 1)];  // beyond K: any value, times zero
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) xb[s] = read_x(0, 4 * g + s);
      }
      if constexpr (!kHFirst) read_h();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (next < end) request(next);
      const int nsp = w == 3 ? sp + nw : sp, nwv = (w + 1) & 3;
      if constexpr (GATHER) {
        if (nsp < end_split && chunk_of(nsp, nwv) < chunks_end(nsp)) request_chain(nsp, nwv);
      }
      if constexpr (!kHFirst) multiply_h();
      if constexpr (GATHER) {
        if (sp < end_split && w == 3 && i < kTokens) {
#pragma unroll
          for (int a = 0; a < NT; ++a)
            *reinterpret_cast<f32x4_t*>(split_sums + ((sp - first_split) * NT + a) * kTokens * 64 + (g * kTokens + i) * 16) = ah[a][0][0][0];
        }
        sp = __builtin_amdgcn_readfirstlane(nsp);
        w = __builtin_amdgcn_readfirstlane(nwv);
      }
      if (has) {
        if (half) {  // nothing of its second half counts, whatever lies there
#pragma unroll
          for (int s = 0; s < 4; ++s) xb[s] = g >= 2 ? u32x4_t{0, 0, 0, 0} : xb[s];
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) sc[rt] = g >= 2 ? 0.f : sc[rt];
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          uint32_t pairs[4][4];  // all reads of a tile's chunk in flight together
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int b = 0; b < 4; ++b) pairs[s][b] = pair_of(cd[rt][s], b);
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            u32x4_t wf;
#pragma unroll
            for (int b = 0; b < 4; ++b) wf[b] = pack_pair(scaled_lo(pairs[s][b], sc[rt]), scaled_hi(pairs[s][b], sc[rt]));
            acc[rt][set % SETS][s] = mfma(wf, xb[s], acc[rt][set % SETS][s]);
          }
        }
      }
      c = next;
    };
    while (c < end || (GATHER && sp < end_split)) {  // a segment is an even number of rounds: sets do not shift
      const int split = c >> 2;
      step(std::integral_constant<int, 0>());
      if constexpr (SETS > 1 || (NT > 0 && kHSets > 1)) {
        if (c < end || (GATHER && sp < end_split)) step(std::integral_constant<int, 1>());
      }
      if constexpr (PAIRED) {  // chains 0 and 1 of the split, or 2 and 3
        if (i < kTokens) {
#pragma unroll
          for (int a = 0; a < NT; ++a) {
            char* const to = split_sums + ((split - first_split) * 3 * NT + a) * kTokens * 64 + (g * kTokens + i) * 16;
            if (wave & 1) {
              *reinterpret_cast<f32x4_t*>(to + NT * kTokens * 64) = ah[a][0][0][0];
              *reinterpret_cast<f32x4_t*>(to + 2 * NT * kTokens * 64) = ah[a][0][1][0];
            } else {
              *reinterpret_cast<f32x4_t*>(to) = ah[a][0][0][0] + ah[a][0][1][0];
            }
          }
        }
      }
    }
    if constexpr (SPLITS) {
      __syncthreads();  // the segment's splits are in LDS
#pragma unroll
      for (int j = 0; j < kHOwn; ++j) {
        const int e = t + j * 64 * MAXW;
        if (e < kHElements) {
          const float* const from = reinterpret_cast<const float*>(split_sums) + e;
          constexpr int kSums = few_split_sums(FORM);
          int n = end_split - first_split;
          const bool last_of_one = PAIRED && 4 * (end_split - 1) + 1 >= n_chunks;  // the last split has no third and fourth chain
          if (last_of_one) --n;
#pragma unroll 4
          for (int q = 0; q < n; ++q) {
            float sum = from[kSums * q * kHElements];
            if constexpr (PAIRED) sum = (sum + from[(3 * q + 1) * kHElements]) + from[(3 * q + 2) * kHElements];
            h_sum[j] += sum;
          }
          if (last_of_one) h_sum[j] += from[kSums * n * kHElements];
        }
      }
    }
    first += seg_chunks;
    if (first >= n_chunks) break;
    __syncthreads();  // every wave is done with the segment's scalers (and splits)
    request_scalers(first * 2, KB - 2 * first < (kSegment >> 6) ? KB - 2 * first : kSegment >> 6);
    if (first + start < n_chunks) request(first + start);
    if constexpr (GATHER) {
      if (first / seg_chunks * seg_splits + wave < n_splits) request_chain(first / seg_chunks * seg_splits + wave, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  }

  // ---- the parts of the sums meet in LDS, [part][tile][lane][v] at the head of each wave's stage, and are added in order
  constexpr int kSteps = NA > 0 ? (NA + 1) / 2 : 2;  // MFMA steps of the adapter, 32 ranks each (the ranks of a group add up to at most 64)
  u32x4_t bv[RT][kSteps], hv[PAIR ? 2 : 1][kSteps];  // wave 0: ranks 32 q + 8 g .. + 7 of its rows' lora_b and of its token's h
  if (wave == 0) {
#pragma unroll
    for (int q = 0; q < kSteps; ++q) {
      const int r = 32 * q + 8 * g;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        bv[rt][q] = u32x4_t{0, 0, 0, 0};
        if (r < member(rt).R) bv[rt][q] = *reinterpret_cast<const u32x4_t*>(member(rt).lora_b + (int64_t)(first_row(rt) + i) * member(rt).R + r);
      }
      if constexpr (NA == 0) {
#pragma unroll
        for (int u = 0; u < (PAIR ? 2 : 1); ++u) {
          hv[u][q] = u32x4_t{0, 0, 0, 0};
          if (i < M && r < member(u).R) hv[u][q] = *reinterpret_cast<const u32x4_t*>(member(u).h + (int64_t)i * member(u).ldh + r);
        }
      }
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int u = 0; u < SETS; ++u)
#pragma unroll
      for (int s = 1; s < 4; ++s) acc[rt][u][0] += acc[rt][u][s];
  auto leave = [&](int u, int rt) { *reinterpret_cast<f32x4_t*>(stage + (u * RT + rt) * 1024 + lane * 16) = acc[rt][u][0]; };
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int u = 0; u < SETS; ++u)
      if (u > 0 || wave > 0) leave(u, rt);
  if constexpr (NT > 0) {
    // h in bf16, [rank tile][token][16 ranks], over the code table (every wave is past its last chunk)
    char* const h_tile = few_smem;
    static_assert(NT * 16 * 32 <= few_lut_bytes(NT), "h lies where the code table was");
    auto h_done = [&](int e, float sum) {  // element e of [rank tile][4 ranks][token][4]
      const int a = e / (16 * kTokens), token = (e >> 2) & (kTokens - 1), r = 4 * ((e / (4 * kTokens)) & 3) + (e & 3);
      const uint16_t bits = f32_to_bf16_bits(sum);
      *reinterpret_cast<uint16_t*>(h_tile + (a * 16 + token) * 32 + r * 2) = bits;
      const SmallMArgs& ma = member(a / NA);
      const int rank = 16 * (a % NA) + r;
      if (ma.h_out && wg == 0 && token < M && rank < ma.R) ma.h_out[(int64_t)token * ma.ldh + rank] = bits;
    };
    if constexpr (SPLITS) {
#pragma unroll
      for (int j = 0; j < kHOwn; ++j)
        if (t + j * 64 * MAXW < kHElements) h_done(t + j * 64 * MAXW, h_sum[j]);
    } else {
      // part 2 wave + b + 8 u of sixteen, behind the wave's partial sums
      constexpr int kAt = SETS * RT * 1024;
      static_assert(kAt + kHSets * 2 * kHElements * 4 <= kStage, "the parts of h fit a stage");
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int u = 0; u < kHSets; ++u)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            if (i < kTokens)
              *reinterpret_cast<f32x4_t*>(stage + kAt + ((u * 2 + b) * kHElements + a * 16 * kTokens) * 4 + (g * kTokens + i) * 16) = ah[a][u][b][0] + ah[a][u][b][1];
      __syncthreads();
      const int parts = KB < 16 ? KB : 16;
      for (int e = t; e < kHElements; e += blockDim.x) {
        auto part = [&](int q) {
          const int from = (q % (2 * MAXW)) >> 1, slot = 2 * (q / (2 * MAXW)) + (q & 1);
          return *reinterpret_cast<const float*>(stages + from * kStage + kAt + (slot * kHElements + e) * 4);
        };
        float sum = part(0);
        if (parts == 16) {
#pragma unroll
          for (int q = 1; q < 16; ++q) sum += part(q);
        } else {
          for (int q = 1; q < parts; ++q) sum += part(q);
        }
        h_done(e, sum);
      }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int u = 0; u < (PAIR ? 2 : 1); ++u)
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
          const int r = 32 * q + 8 * g;
          hv[u][q] = u32x4_t{0, 0, 0, 0};
          if (i < M && r < member(u).R) hv[u][q] = *reinterpret_cast<const u32x4_t*>(h_tile + ((u * NA + (r >> 4)) * 16 + i) * 32 + (r & 15) * 2);
        }
    }
  }
  if (wave == 0) {
    // adapter: sum_r bf16(h[m][r] * lscale) * lora_b[n][r], the operands the large-M kernel feeds its MFMA
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const float ls = member(rt).lscale;
#pragma unroll
      for (int q = 0; q < kSteps; ++q) {
        if (32 * q >= member(rt).R) break;
        u32x4_t h;
#pragma unroll
        for (int d = 0; d < 4; ++d) h[d] = pack_pair(lo_of(hv[PAIR ? rt & 1 : 0][q][d]) * ls, hi_of(hv[PAIR ? rt & 1 : 0][q][d]) * ls);
        acc[rt][0][0] = mfma(bv[rt][q], h, acc[rt][0][0]);
      }
      leave(0, rt);
    }
  }
  __syncthreads();
  // every thread finishes one output (PAIR: one of each member) at a time: one wave alone took 1.3 us over sixteen waves' sums
  const int parts = SETS * MAXW < n_chunks ? SETS * MAXW : n_chunks;
  for (int e = t; e < 256 * (PAIR ? RT / 2 : RT); e += blockDim.x) {
    const int tile = e >> 8, token = (e >> 2) & 15, row = 4 * ((e >> 6) & 3) + (e & 3);
    if (token >= M) continue;
    uint32_t out[PAIR ? 2 : 1];
#pragma unroll
    for (int u = 0; u < (PAIR ? 2 : 1); ++u) {
      const int rt = PAIR ? 2 * tile + u : tile;
      const SmallMArgs& a = member(u);
      const int n = first_row(rt) + row;
      auto part = [&](int q) {
        const int from = PAIRED ? 2 * (q >> 2) + (q & 1) : q % MAXW, set = PAIRED ? (q >> 1) & 1 : q / MAXW;
        return *reinterpret_cast<const float*>(stages + from * kStage + (set * RT + rt) * 1024 + (e & 255) * 4);
      };
      float o = part(0);
      if (parts == SETS * MAXW) {
#pragma unroll
        for (int q = 1; q < SETS * MAXW; ++q) o += part(q);
      } else {
        for (int q = 1; q < parts; ++q) o += part(q);
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

// Launch shape at most 16 tokens.  The waves and their sets fix the order in which a row's products are summed (parts of four
// chains: sixteen up to 4096 rows and, below 8192, where the layer is no wider than its input, four beyond 12288 rows over
// less than 8192 columns, otherwise eight) and depend on the layer alone, so that a row gets the same bits alone, in a
// batch of up to 16 tokens and inside a group; row tiles do not enter the sums.  Measured over 27 layers of 256 - 28672 rows
// and 1024 - 28672 columns (us, weights from HBM, launch gap included):
//  * eight waves (4096 x 4096 at 1 / 13 tokens, h in the launch's own order: four 8.7 / 9.3, eight 6.7 / 7.9, sixteen 7.6 / 8.8; 2048 x 8192
//    at 13: 14.6 / 11.1 / 12.3), four where the layer has workgroups to spare and a short contraction (gate / up pair of 14336 x 4096,
//    eight and four: 21.8 and 20.6);
//  * two row tiles, which share the reads of x and lora_a, from 8192 rows on (8192 x 2048 at 13 tokens: one 7.9, two 7.0; 14336 x 4096 at one
//    token with its h, in the launch's own order: 17.8 and 14.9), but one where four waves at a few tokens read h instead (the
//    same layer 13.9, two 16.1).
struct FewConfig {
  int rt, waves, sets;
  bool operator==(const FewConfig& o) const { return rt == o.rt && waves == o.waves && sets == o.sets; }
};
int few_waves(int64_t N, int64_t K) { return N > 12288 && K < 8192 ? 4 : 8; }
int few_sets(int64_t N, int64_t K) { return N <= 4096 || (N < 8192 && N <= K) ? 2 : 1; }
FewConfig few_config(int64_t M, int64_t N, int64_t K, bool hidden) {
  const int waves = few_waves(N, K);
  return {N >= 8192 && (hidden || waves == 8 || M > 4) ? 2 : 1, waves, few_sets(N, K)};
}
FewConfig few_pair_config(int64_t N, int64_t K, bool hidden) {
  const int waves = few_waves(N, K);
  return {hidden && waves == 4 ? 4 : 2, waves, few_sets(N, K)};
}
constexpr int kFewMostLds = 160 * 1024;
HiddenForm few_form(const FewConfig& c, int64_t K) {
  const HiddenOrder o = hidden_order(K);
  return o.splits == 0 ? kWaves : c.sets == 2 && o.chunks_per_split == 8 ? kPaired : kGather;
}
// Whether a launch of these workgroups forms its members' h = x . lora_a^T itself, instead of a launch or two ahead of it; the
// bits are the same.  Every workgroup then reads its members' lora_a, rank_tiles tiles of 16 ranks: up to 128 MiB for the launch
// the better way (us with its h, against reading it, at one token: 8192 x 8192, 128 MiB, 18.3 and 19.2, 4096 x 14336 19.3 and 21.1; at
// 13 tokens 21.3 and 20.0, 23.3 and 22.2, but two launches fewer), not beyond (4096 x 20480, 160 MiB, 26.2 and 25.4, 10240 x 8192
// 30.0 and 23.9, 8192 x 12288, 192 MiB, 25.8 and 24.2); several tiles only where the LDS they take leaves room for every
// workgroup at once (gate / up pair of 8192 x 2048, 512 workgroups in two rounds: 15.1 against 12.1; in one round, 2816 x 1024:
// 7.3 against 9.3).  In the order of the adapters' launch h takes 0.4 us of a launch more over 2048 columns and 1 - 3.5 over
// 4096 - 14336 than in the order that suits the launch (4096 x 4096 6.9 -> 7.9, 2048 x 8192 9.1 -> 11.2; reading it 11.1 and 13.4);
// the gate / up pair of 14336 x 4096 takes 31.0 with it and 27.3 with two launches ahead, in a layer outside a graph 77 and 82.
bool few_hidden(int64_t workgroups, const FewConfig& c, int rank_tiles, int64_t M, int64_t K) {
  const HiddenForm form = few_form(c, K);
  const int mq = M <= 4 ? 1 : 4, segment = few_segment(c.rt, rank_tiles, mq, form);
  // the launch is there for every contraction or for none (launch_few)
  if (few_bytes(c.rt, c.sets, rank_tiles, mq, form, segment, segment / 512, c.waves) > kFewMostLds) return false;
  const int n_chunks = (int)((K + 127) >> 7), waves = n_chunks < c.waves ? n_chunks : c.waves;
  const int bytes = few_bytes(c.rt, c.sets, rank_tiles, mq, form, (int)K, hidden_order(K).splits, waves);
  if (rank_tiles > 1 && workgroups > 256 * (kFewMostLds / bytes)) return false;
  return workgroups * rank_tiles * 32 * K <= int64_t(128) << 20;
}

template <int RT, int MAXW, int SETS, int MQ, int NA, int FORM, bool PAIR, bool ONE>
int launch_few(const SmallMGroup& g, unsigned wgs, uint16_t* act, hipStream_t s) {
  constexpr int NT = NA * (PAIR ? 2 : 1);
  const int K = g.m[0].K, n_chunks = (K + 127) >> 7, waves = n_chunks < MAXW ? n_chunks : MAXW;
  constexpr int kSegment = few_segment(RT, NT, MQ, FORM);
  constexpr int kMost = few_bytes(RT, SETS, NT, MQ, FORM, kSegment, kSegment / 512, MAXW);
  static_assert(kMost <= kFewMostLds, "the LDS of a CU");
  static bool attr_set[64] = {};  // the LDS limit is a per-device attribute of the function
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (dev < 0 || !attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&nf4_few_kernel<RT, MAXW, SETS, MQ, NA, FORM, PAIR, ONE>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kMost);
    if (e != hipSuccess) return fail(TTAMD_ELAUNCH, "nf4_few: cannot reserve %d bytes of LDS: %s", kMost, hipGetErrorString(e));
    if (dev >= 0) attr_set[dev] = true;
  }
  nf4_few_kernel<RT, MAXW, SETS, MQ, NA, FORM, PAIR, ONE>
      <<<dim3(wgs), dim3(64 * waves), few_bytes(RT, SETS, NT, MQ, FORM, K, g.splits, waves), s>>>(g, act);
  return check_launch("nf4_few");
}

template <int RT, int MAXW, int SETS, int MQ, int NA, int FORM>
int launch_few_members(SmallMGroup& g, hipStream_t s) {
  int wgs = 0;
  for (int i = 0; i < g.n; ++i) {
    wgs += g.m[i].N / (16 * RT);
    g.wg_end[i] = wgs;
  }
  return g.n == 1 ? launch_few<RT, MAXW, SETS, MQ, NA, FORM, false, true>(g, wgs, nullptr, s)
                  : launch_few<RT, MAXW, SETS, MQ, NA, FORM, false, false>(g, wgs, nullptr, s);
}

// The shapes that few_config and few_form give.  NA: rank tiles of a member, where the launch forms h.
template <int MQ, int NA, int FORM>
int dispatch_few_members(SmallMGroup& g, const FewConfig& c, hipStream_t s) {
  if (c.rt == 1 && c.sets == 2) return launch_few_members<1, 8, 2, MQ, NA, FORM>(g, s);
  if constexpr (FORM == kPaired) {
    return fail(TTAMD_EUNSUPPORTED, "nf4_few: no such launch");
  } else {
    if (c.rt == 1) {
      if constexpr (MQ == 1 && NA == 0) {
        if (c.waves == 4) return launch_few_members<1, 4, 1, MQ, NA, FORM>(g, s);
      }
      return launch_few_members<1, 8, 1, MQ, NA, FORM>(g, s);
    }
    if constexpr (MQ == 4 || NA > 0) {
      if (c.waves == 4) return launch_few_members<2, 4, 1, MQ, NA, FORM>(g, s);
    }
    if constexpr (MQ == 4 && NA == 2 && FORM == kGather)
      return fail(TTAMD_EUNSUPPORTED, "nf4_few: no room for the operands of h");  // few_hidden
    else
      return launch_few_members<2, 8, 1, MQ, NA, FORM>(g, s);
  }
}
template <int NA>
int dispatch_few_forming(SmallMGroup& g, const FewConfig& c, hipStream_t s) {
  const bool one = g.m[0].M <= 4;  // group of four tokens
  switch (few_form(c, g.m[0].K)) {
    case kWaves: return one ? dispatch_few_members<1, NA, kWaves>(g, c, s) : dispatch_few_members<4, NA, kWaves>(g, c, s);
    case kPaired: return one ? dispatch_few_members<1, NA, kPaired>(g, c, s) : dispatch_few_members<4, NA, kPaired>(g, c, s);
    default: return one ? dispatch_few_members<1, NA, kGather>(g, c, s) : dispatch_few_members<4, NA, kGather>(g, c, s);
  }
}
// rank_tiles: of a member, where the launch forms h; 0 where it reads it
int dispatch_few(SmallMGroup& g, const FewConfig& c, int rank_tiles, hipStream_t s) {
  if (rank_tiles == 0) return g.m[0].M <= 4 ? dispatch_few_members<1, 0, kReads>(g, c, s) : dispatch_few_members<4, 0, kReads>(g, c, s);
  return rank_tiles == 1 ? dispatch_few_forming<1>(g, c, s) : dispatch_few_forming<2>(g, c, s);
}
template <int MQ>
int dispatch_few_pair_reading(const SmallMGroup& g, const FewConfig& c, unsigned wgs, uint16_t* act, hipStream_t s) {
  if (c.waves == 4) return launch_few<2, 4, 1, MQ, 0, kReads, true, false>(g, wgs, act, s);
  return c.sets == 2 ? launch_few<2, 8, 2, MQ, 0, kReads, true, false>(g, wgs, act, s) : launch_few<2, 8, 1, MQ, 0, kReads, true, false>(g, wgs, act, s);
}
// few_pair_forms: more than four tokens only over short contractions, and not with four row tiles
template <int FORM>
int dispatch_few_pair_forming(const SmallMGroup& g, const FewConfig& c, unsigned wgs, uint16_t* act, hipStream_t s) {
  if constexpr (FORM == kWaves) {
    if (g.m[0].M > 4) return c.sets == 2 ? launch_few<2, 8, 2, 4, 1, FORM, true, false>(g, wgs, act, s) : launch_few<2, 8, 1, 4, 1, FORM, true, false>(g, wgs, act, s);
  }
  if (c.sets == 2) return launch_few<2, 8, 2, 1, 1, FORM, true, false>(g, wgs, act, s);
  if constexpr (FORM == kPaired)
    return fail(TTAMD_EUNSUPPORTED, "nf4_few: no such launch");
  else
    return c.rt == 4 ? launch_few<4, 4, 1, 1, 1, FORM, true, false>(g, wgs, act, s) : launch_few<2, 8, 1, 1, 1, FORM, true, false>(g, wgs, act, s);
}
bool few_pair_forms(const FewConfig& c, int64_t M, int64_t K) { return M <= 4 || (c.rt == 2 && few_form(c, K) == kWaves); }
int dispatch_few_pair(const SmallMGroup& g, const FewConfig& c, bool hidden, uint16_t* act, hipStream_t s) {
  const unsigned wgs = g.m[0].N / (8 * c.rt);
  if (!hidden) return g.m[0].M <= 4 ? dispatch_few_pair_reading<1>(g, c, wgs, act, s) : dispatch_few_pair_reading<4>(g, c, wgs, act, s);
  switch (few_form(c, g.m[0].K)) {
    case kWaves: return dispatch_few_pair_forming<kWaves>(g, c, wgs, act, s);
    case kPaired: return dispatch_few_pair_forming<kPaired>(g, c, wgs, act, s);
    default: return dispatch_few_pair_forming<kGather>(g, c, wgs, act, s);
  }
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
  if (gg.M > kFewTokens || gg.K >= kFewMaxK || hidden_order(gg.K).chunks_per_split > 8) return false;
  for (int i = 0; i < gg.n; ++i)
    if (gg.rank[i] < 8 || gg.rank[i] > kFewHiddenRank) return false;
  if (gated) {
    const FewConfig c = few_pair_config(gg.N[0], gg.K, true);
    return rank_tiles_of(gg, 0, 2) == 1 && few_pair_forms(c, gg.M, gg.K) && few_hidden(gg.N[0] / (8 * c.rt), c, 2, gg.M, gg.K);
  }
  for (int i = 0; i < gg.n;) {
    const int j = run_of(gg, i, [&](int p, int q) { return same_few(gg, p, q, true); });
    const FewConfig c = few_config(gg.M, gg.N[i], gg.K, true);
    int64_t wgs = 0;
    for (int q = i; q < j; ++q) wgs += gg.N[q] / (16 * c.rt);
    if (!few_hidden(wgs, c, rank_tiles_of(gg, i, j), gg.M, gg.K)) return false;
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
  const HiddenOrder order = hidden_order(gg.K);
  SmallMGroup g = {};
  g.splits = order.splits;
  g.chunks_per_split = order.chunks_per_split;
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
