// y = x . D(W)^T (+ bias) + scale . h . lora_b^T, times an optional column scale, for a handful of tokens (M <= 64):
// the decode / evaluation regime of linear_nf4 and LoRALinear.forward (torchtune/modules/peft/lora.py:128-147,
// torchtune/modules/low_precision/nf4_linear.py:56-70).
//
// With so few rows the work is streaming the packed weight once: 0.5625 bytes per weight element against 2 for a
// dense bf16 weight.  A workgroup owns 16 or 32 weight rows and the whole contraction, expands the codes in registers
// exactly as the large-M kernel does (byte -> fp32 pair from an LDS table, times the fp32 block scaler, one rounding to
// bf16 - the bits of ttamd_nf4_dequantize) and feeds v_mfma_f32_16x16x32_bf16 with the weight rows as the row operand
// and 16-token tiles of x as the column operand.  A lane reads 16 contiguous bytes of codes (32 elements of
// its row: the four lane groups of a row cover one 64-byte piece) and uses one dword of them per MFMA; x is small and
// comes from the cache.  The waves' partial sums meet in LDS in a fixed order.
//
//  * nf4_few_kernel (at most 16 tokens, generation): the waves take 128-wide chunks of K in turn, one chunk each at a
//    time.  Neighbouring waves then read neighbouring pieces of the same rows; groups of four chunks per wave, which
//    put more bytes in flight, were slower at every size.  Only the lanes of tokens that exist ask for x.  The adapter
//    is one more MFMA step whose operands are requested ahead of the loop, and the gate / up pair of a feed-forward
//    shares a workgroup, so that silu(gate) * up leaves the same launch.
//  * nf4_small_m_kernel (17 - 64 tokens): groups of U chunks per wave, two or four token tiles.
#include "common.h"
#include "group.h"
#include "nf4_math.h"
#include "swiglu_math.h"

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

// RT tiles of 16 weight rows per workgroup, at most MAXW waves.  PAIR: tile 0 belongs to grp.m[0] (gate), tile 1 to grp.m[1]
// (up projection, the same width), and act = bf16(bf16(silu(y_0)) * y_1) is written as well.
// ONE: the launch has one member, and its arguments sit at fixed places (found through `which` they cost two dependent
// scalar loads before the first request: 0.4 us of a launch of 6 - 8).
template <int RT, int MAXW, bool PAIR, bool ONE>
__global__ __launch_bounds__(64 * MAXW) void nf4_few_kernel(const SmallMGroup grp, uint16_t* __restrict__ act) {
  static_assert(!PAIR || RT == 2, "a pair is two row tiles");
  int which = 0;  // uniform over the workgroup
  if constexpr (!PAIR && !ONE) {
#pragma unroll
    for (int q = 0; q < kGroupMax - 1; ++q)
      if (q < grp.n - 1 && (int)blockIdx.x >= grp.wg_end[q]) which = q + 1;
  }
  __shared__ float2 lut[256];
  __shared__ float red[(MAXW - 1) * RT * 256];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nw = blockDim.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int M = grp.m[which].M, K = grp.m[which].K;
  const int wg = (int)blockIdx.x - (!PAIR && !ONE && which ? grp.wg_end[which - 1] : 0);
  auto member = [&](int rt) -> const SmallMArgs& { return grp.m[PAIR ? rt : which]; };
  auto first_row = [&](int rt) { return PAIR ? 16 * wg : 16 * (RT * wg + rt); };  // N % (16 RT) == 0: every row exists

  const bool token = i < M;
  const uint16_t* xrow = grp.m[which].x + (int64_t)(token ? i : 0) * K + 32 * g;
  const uint8_t* crow[RT];
  const float* srow[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int64_t n = first_row(rt) + i;
    crow[rt] = member(rt).codes + ((n * K) >> 1) + 16 * g;
    srow[rt] = member(rt).bscal + n * (K >> 6) + (g >> 1);
  }
  u32x4_t cd[RT], xb[4];
  float sc[RT];
  auto request = [&](int c) {
    const bool in = c * 128 + 32 * g < K;  // the last chunk of a K that is an odd multiple of 64 is half a chunk
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      cd[rt] = u32x4_t{0, 0, 0, 0};
      sc[rt] = 0.f;
      if (in) {
        cd[rt] = *reinterpret_cast<const u32x4_t*>(crow[rt] + (int64_t)c * 64);
        sc[rt] = srow[rt][2 * c];
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      xb[s] = u32x4_t{0, 0, 0, 0};
      if (in && token) xb[s] = *reinterpret_cast<const u32x4_t*>(xrow + c * 128 + 8 * s);
    }
  };
  const int n_chunks = (K + 127) >> 7;
  // The first chunk and wave 0's adapter operands are asked for before the code table is built: a workgroup lives for
  // little more than one trip to memory, and neither the table nor a second trip at the end must stand in its way.
  int c = wave;
  if (c < n_chunks) request(c);
  auto adapter = [&](int rt, int r0, u32x4_t& hv, u32x4_t& bv) {  // ranks r0 + 8 g .. + 7 (R % 8 == 0)
    const SmallMArgs& a = member(rt);
    hv = bv = u32x4_t{0, 0, 0, 0};
    if (r0 + 8 * g < a.R) {
      bv = *reinterpret_cast<const u32x4_t*>(a.lora_b + (int64_t)(first_row(rt) + i) * a.R + r0 + 8 * g);
      if (token) hv = *reinterpret_cast<const u32x4_t*>(a.h + (int64_t)i * a.ldh + r0 + 8 * g);
    }
  };
  u32x4_t hv[RT], bv[RT];
  if (wave == 0) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) adapter(rt, 0, hv[rt], bv[rt]);
  }
  for (int e = t; e < 256; e += blockDim.x)
    lut[e] = make_float2(round_to_bf16(nf4_code_value(e >> 4)), round_to_bf16(nf4_code_value(e & 15)));
  f32x4_t acc[RT][4];  // four chains
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int s = 0; s < 4; ++s) acc[rt][s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  while (c < n_chunks) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        u32x4_t wf;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const float2 p = lut[(cd[rt][s] >> (8 * b)) & 0xffu];
          wf[b] = pack_pair(p.x * sc[rt], p.y * sc[rt]);
        }
        acc[rt][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf), __builtin_bit_cast(bf16x8_t, xb[s]),
                                                             acc[rt][s], 0, 0, 0);
      }
    c += nw;
    if (c < n_chunks) request(c);
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
    for (int s = 1; s < 4; ++s) acc[rt][0] += acc[rt][s];
    if (wave == 0) {
      // adapter: sum_r bf16(h[m][r] * lscale) * lora_b[n][r], the operands the large-M kernel feeds its MFMA
      const float ls = member(rt).lscale;
      for (int r0 = 0; r0 < member(rt).R; r0 += 32) {
        if (r0 > 0) adapter(rt, r0, hv[rt], bv[rt]);
        u32x4_t hs;
#pragma unroll
        for (int d = 0; d < 4; ++d) hs[d] = pack_pair(lo_of(hv[rt][d]) * ls, hi_of(hv[rt][d]) * ls);
        acc[rt][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, bv[rt]), __builtin_bit_cast(bf16x8_t, hs),
                                                             acc[rt][0], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) red[((wave - 1) * RT + rt) * 256 + v * 64 + lane] = acc[rt][0][v];
    }
  }
  __syncthreads();
  if (wave != 0) return;
  // acc[rt][0][v] = the wave's share of y[i][first_row(rt) + 4 g + v]
  u32x2_t out[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const SmallMArgs& a = member(rt);
    const int nb = first_row(rt) + 4 * g;
    float o[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      o[v] = acc[rt][0][v];
      for (int w = 0; w < nw - 1; ++w) o[v] += red[(w * RT + rt) * 256 + v * 64 + lane];
    }
    if (a.bias) {
      const u32x2_t bb = *reinterpret_cast<const u32x2_t*>(a.bias + nb);
      o[0] += lo_of(bb.x); o[1] += hi_of(bb.x); o[2] += lo_of(bb.y); o[3] += hi_of(bb.y);
    }
    if (a.cscale) {
      const u32x2_t cc = *reinterpret_cast<const u32x2_t*>(a.cscale + nb);
      o[0] *= lo_of(cc.x); o[1] *= hi_of(cc.x); o[2] *= lo_of(cc.y); o[3] *= hi_of(cc.y);
    }
    out[rt].x = pack_pair(o[0], o[1]);
    out[rt].y = pack_pair(o[2], o[3]);
    if (token) *reinterpret_cast<u32x2_t*>(a.y + (int64_t)i * a.N + nb) = out[rt];
  }
  if constexpr (PAIR) {
    u32x2_t p;
    p.x = swiglu_gate_pair(out[0].x, out[1].x);
    p.y = swiglu_gate_pair(out[0].y, out[1].y);
    if (token) *reinterpret_cast<u32x2_t*>(act + (int64_t)i * grp.m[0].N + 16 * wg + 4 * g) = p;
  }
}

// Launch shape at most 16 tokens.  The waves fix the order in which a row's products are summed and depend on the
// layer alone, so that a row gets the same bits alone, in a batch of up to 16 tokens and inside a group; row tiles do not
// enter the sums.  Measured over 48 layers of 256 - 28672 rows and 1024 - 28672 columns (us, weights from HBM, launch gap included):
//  * up to 4096 rows a CU has one workgroup, which wants all the waves: one token, sixteen and eight waves: 4096 x 4096 7.5 and 7.9,
//    4096 x 14336 15.8 and 18.9.  Layers below 8192 rows that are no wider than their input keep sixteen, too: a query projection
//    then shares a launch with its key / value members.
//  * up to 12288 rows eight: one token, sixteen / eight / four: 6912 x 2560 9.4 / 7.7 / 8.7, 8192 x 8192 18.9 / 17.1 / 22.0, 12288 x 2048
//    11.3 / 7.9 / 8.5.  With two row tiles, which halve the reads of x, where those weigh and the layer is no wider than 8192 (16
//    tokens, one and two tiles: 8192 x 28672 83.8 and 58.8, 8192 x 4096 14.8 and 13.4, but 8192 x 2048 9.1 and 9.9; 12 tokens, 12288 x 4096
//    18.4 and 19.5).
//  * beyond, three workgroups of eight waves per CU do not hold the layer any more: four (one token, eight and four: 14336 x 4096
//    17.0 and 15.6, 16384 x 1024 7.9 and 6.9), unless the contraction is long (28672 x 8192 46.8 and 49.3); two tiles from 5 tokens on
//    where x is large enough (14336 x 4096 at 8 tokens 21.2 and 18.4, 16384 x 1024 7.7 and 8.7).
struct FewConfig {
  int rt, waves;
  bool operator==(const FewConfig& o) const { return rt == o.rt && waves == o.waves; }
};
FewConfig few_config(int64_t M, int64_t N, int64_t K) {
  if (N <= 4096 || (N < 8192 && N <= K)) return {1, 16};
  if (N <= 12288) return {N <= 8192 && M * K >= 40960 ? 2 : 1, 8};
  return {M > 4 && M * K >= 16384 ? 2 : 1, K < 8192 ? 4 : 8};
}

template <int RT, int MAXW, bool PAIR>
int launch_few(SmallMGroup& g, void* act, hipStream_t s) {
  int wgs = 0;
  for (int i = 0; i < (PAIR ? 1 : g.n); ++i) {
    wgs += g.m[i].N / (PAIR ? 16 : 16 * RT);
    g.wg_end[i] = wgs;
  }
  const int n_chunks = (g.m[0].K + 127) >> 7;
  const dim3 grid((unsigned)wgs), block(64 * (n_chunks < MAXW ? n_chunks : MAXW));
  if (!PAIR && g.n == 1)
    nf4_few_kernel<RT, MAXW, PAIR, true><<<grid, block, 0, s>>>(g, nullptr);
  else
    nf4_few_kernel<RT, MAXW, PAIR, false><<<grid, block, 0, s>>>(g, reinterpret_cast<uint16_t*>(act));
  return check_launch("nf4_few");
}

int dispatch_few(SmallMGroup& g, const FewConfig& c, void* pair_act, hipStream_t s) {
  if (pair_act) {
    if (c.waves == 16) return launch_few<2, 16, true>(g, pair_act, s);
    return c.waves == 8 ? launch_few<2, 8, true>(g, pair_act, s) : launch_few<2, 4, true>(g, pair_act, s);
  }
  if (c.waves == 16) return launch_few<1, 16, false>(g, nullptr, s);
  if (c.waves == 8) return c.rt == 2 ? launch_few<2, 8, false>(g, nullptr, s) : launch_few<1, 8, false>(g, nullptr, s);
  return c.rt == 2 ? launch_few<2, 4, false>(g, nullptr, s) : launch_few<1, 4, false>(g, nullptr, s);
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
  if (M <= kFewTokens) return dispatch_few(g, few_config(M, N, K), nullptr, s);
  return dispatch_small_m(g, small_m_config(M, N, K), s);
}

// The members of a group (same x, M, K) in as few launches as their launch shapes allow: consecutive members with
// the same shape share one.  act != nullptr (two members of equal width): *act_done says whether the launch wrote
// act = silu(y_0) * y_1 too.
int run_small_m_group(const void* x, const GroupGemm& gg, const void* h_cat, void* act, bool* act_done, hipStream_t s) {
  TT_REQUIRE(gg.M > 0 && gg.M <= small_m_limit(), "nf4_small_m: M (%lld) out of range", (long long)gg.M);
  SmallMArgs all[kGroupMax] = {};
  for (int j = 0; j < gg.n; ++j) {
    TT_REQUIRE(gg.N[j] / 16 < (int64_t(1) << 27) && gg.N[j] * gg.K < (int64_t(1) << 40), "nf4_small_m: weight too large");
    SmallMArgs& a = all[j];
    a.x = reinterpret_cast<const uint16_t*>(x);
    a.codes = gg.codes[j];
    a.bscal = gg.bscal[j];
    a.h = reinterpret_cast<const uint16_t*>(h_cat) + gg.r_off[j];
    a.lora_b = gg.lora_b[j];
    a.bias = gg.bias[j];
    a.y = gg.y[j];
    a.M = (int)gg.M; a.N = (int)gg.N[j]; a.K = (int)gg.K; a.R = gg.rank[j]; a.ldh = gg.r_off[gg.n];
    a.lscale = gg.scale[j];
  }
  const bool few = gg.M <= kFewTokens;
  if (act && few && gg.n == 2 && gg.N[0] == gg.N[1]) {
    SmallMGroup g = {};
    g.m[0] = all[0];
    g.m[1] = all[1];
    g.n = 2;
    *act_done = true;
    return dispatch_few(g, few_config(gg.M, gg.N[0], gg.K), act, s);
  }
  int i = 0;
  while (i < gg.n) {
    SmallMGroup g = {};
    int j = i;
    auto same = [&](int q) {
      return few ? few_config(gg.M, gg.N[q], gg.K) == few_config(gg.M, gg.N[i], gg.K)
                 : small_m_config(gg.M, gg.N[q], gg.K) == small_m_config(gg.M, gg.N[i], gg.K);
    };
    for (; j < gg.n && same(j); ++j) g.m[j - i] = all[j];
    g.n = j - i;
    if (int rc = few ? dispatch_few(g, few_config(gg.M, gg.N[i], gg.K), nullptr, s) : dispatch_small_m(g, small_m_config(gg.M, gg.N[i], gg.K), s))
      return rc;
    i = j;
  }
  return TTAMD_OK;
}

}  // namespace ttamd
