// Fused NF4-dequantise + bf16 MFMA products of a few dozen to some thousand rows:
//
//     C[M, Nout] = X[M, Kc] . D(Wv)[Nout, Kc]^T  (+ bias)  + (lscale . lX)[M, R] . lW[Nout, R]^T
//
// (the operands, the weight views of forward and grad-input and the scaler modes are those of nf4_gemm_rs.hip, which has the
// rules that send a product here or elsewhere).
//
// Eight waves on a tile of 64 x 128 (KG = 4), 96 x 256 or 128 x 256 (KG = 2).  A step is 32 KG contraction indices, of which wave
// group k of KG multiplies its 32; a wave has 64 columns and all rows of the tile, so a weight is expanded once per tile, and the
// groups' sums meet in LDS at the end.  Activations, codes and scalers reach LDS by direct loads into a ring of three or four
// stages; a wave holds its operands in registers a step ahead.
//
// What bounds it: the vector ALU beside the matrix pipes.  A pair of weights costs four instructions (the table's address, two
// products, one rounding); up to six of them ride under a 32 x 32 x 16 product (two waves per SIMD; a loop of that product
// alone and V others takes 33 cycles a product for V = 0, 36 for 6, 46 for 8; 16 x 16 x 32: 17, 18 for 2, 23 for 3), which is why the
// loop is cut into quarters that mix them evenly, and why the larger shape is taken.  128-row tiles need 4.7 a product: a step of
// 1024 matrix cycles takes 1270; 64-row tiles need 9.4, and a step of 512 matrix cycles takes 1300.
//   * Table reads: a byte's two values are an 8-byte entry in 32 copies, 256 bytes apart, so that no two lanes of a read share
//     a bank and the address is one v_perm_b32 (byte, lane).  With one copy LDS was busy 0.76 of the time, half of it on conflicts.
//   * 64 x 128 tiles: where 128 x 256 tiles would have to be cut into slices to fill the chip, 4 - 16 workgroups left a slab of 128
//     KB each and a second launch added them up.  Whole contractions on small tiles take 16 us for 2048 x 2048 at 700 tokens (five
//     slices: 19 + 5), 25 for 4096 x 4096 at 333 (24 + 6), 8 for 512 x 512 at 100 (12).
//   * 96 x 256 tiles: 448 instead of 336 workgroups where the latter would part-fill a second round, 224 instead of 168.
//   * The adapter's operands are requested ahead of the exchange, the table is built while the first loads are under way.
// Against the kernels that it replaced (128 x 256 tiles on four waves in slices, on two groups of four whole; 1470 products and
// groups of seven model shapes, 33 - 2047 rows): 0.85 of their time on average, 0.74 - 0.83 up to 1000 rows, level near full
// rounds, where the power limit holds both.
#include "common.h"
#include "group.h"
#include "nf4_gemm_args.h"
#include "nf4_math.h"

#include <type_traits>

namespace ttamd {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

__device__ __constant__ float kNF4Mid[16] = TT_NF4_TABLE;

__device__ __forceinline__ uint32_t pack_pair(float lo, float hi) {
  bf16x2_t v;
  v.x = (__bf16)lo;
  v.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, v);
}

#define TT_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

enum MidForm { kPlain = 0, kSegments = 1, kMembers = 2 };

constexpr int kTableBytes = 64 * 1024;  // 256 entries of 256 bytes: 32 copies of a pair of fp32

// MT: groups of 32 rows of a tile; KG: wave groups that share the contraction of a step
template <int MT, int KG>
struct NMid {
  static constexpr int rows = 32 * MT;
  static constexpr int wn = 8 / KG;     // waves side by side, 64 columns each
  static constexpr int cols = 64 * wn;
  static constexpr int step = 32 * KG;  // contraction indices of a step
  static constexpr int a_bytes = rows * step * 2;
  static constexpr int c_bytes = cols * step / 2;  // 8 KiB
  static constexpr int s_bytes = 8 * 256;          // a wave's scalers
  static constexpr int stage = a_bytes + c_bytes + s_bytes;
  static constexpr int stages = (160 * 1024 - kTableBytes) / stage;  // 4 with 96 rows, else 3
  static constexpr int lds = kTableBytes + stages * stage;
  static constexpr int a_wave = a_bytes / 8;                 // bytes of the activation stage that a wave requests
  static constexpr int a_loads = (a_wave + 1023) / 1024, loads = a_loads + 2;  // a wave's loads per step
  // Of its columns' 2 MT squares of 32 x 32 a wave finishes own, nj columns of them and mr rows
  static constexpr int own = 2 * MT / KG, nj = own % 2 ? 1 : 2, mr = own / nj;
  static_assert(a_wave % 512 == 0 && 2 * MT % KG == 0 && stages >= 3 && stages <= 4, "tile");
  static_assert(8 * (KG - 1) * own * 4096 <= lds, "the exchange fits");
  // square e of those that wave group k finishes: its column and row
  static constexpr int sq_j(int k, int e) { return nj == 2 ? e & 1 : own == 1 ? k & 1 : k; }
  static constexpr int sq_i(int k, int e) { return nj == 2 ? k * mr + (e >> 1) : own == 1 ? k >> 1 : e; }
};

template <int MT, int KG, int MODE, int FORM, bool FOLD>
__global__ __launch_bounds__(512, 2) void nf4_gemm_mid_kernel(const RsArgs ga, const std::conditional_t<FORM == kMembers, RsMembers, RsSegs> sg) {
#if defined(__HIP_DEVICE_COMPILE__)
  using S = NMid<MT, KG>;
  constexpr bool SEG = FORM == kSegments;
  static_assert(!SEG || MODE == 1, "segments: grad-input");
  static_assert(FORM != kMembers || MODE == 2, "members: forward");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  RsArgs g = ga;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wv / S::wn, wn = wv % S::wn;
  const int l31 = lane & 31, h = lane >> 5;

  // workgroup ids go round-robin to the 8 XCDs: each gets a run of neighbouring items (of every member: their workgroups take
  // different times)
  const int xcd = (int)(blockIdx.x & 7);
  int slot_of_xcd = (int)(blockIdx.x >> 3);
  if constexpr (FORM == kMembers) {
    int q = 0;
    while (slot_of_xcd >= sg.slot_end[q]) ++q;  // uniform; the grid ends at slot_end[n - 1]
    slot_of_xcd -= q ? sg.slot_end[q - 1] : 0;
    g.per_xcd = sg.slot_end[q] - (q ? sg.slot_end[q - 1] : 0);
    g.codes = sg.codes[q];
    g.scal = sg.scal[q];
    g.lX = sg.lX[q];
    g.lW = sg.lW[q];
    g.bias = sg.bias[q];
    g.C = sg.C[q];
    g.Nout = sg.Nout[q];
    g.R = sg.R[q];
    g.lscale = sg.lscale[q];
    g.tiles_n = (g.Nout + S::cols - 1) / S::cols;
    g.slices = sg.slices[q];
    g.steps = sg.steps[q];
    g.chain = sg.chain[q];
    g.part += sg.part_at[q];
    g.items = g.tiles_m * g.tiles_n * g.slices;
  }
  const int item = xcd * g.per_xcd + slot_of_xcd;
  if (slot_of_xcd >= g.per_xcd || item >= g.items) return;
  // bands of at most four row tiles: the 32 workgroups of an XCD then cover about 4 x 8 tiles, whose operands are the least
  const int bands = (g.tiles_m + 3) >> 2, band_rows = (g.tiles_m + bands - 1) / bands;
  const int slices = g.slices;
  const bool split = slices > 1;
  const int band = item / (band_rows * g.tiles_n * slices);
  const int in_band = item - band * band_rows * g.tiles_n * slices;
  const int rows_here = g.tiles_m - band * band_rows < band_rows ? g.tiles_m - band * band_rows : band_rows;
  const int tile_m = band * band_rows + in_band % rows_here;
  const int rest = in_band / rows_here;
  const int slice = rest % slices, tile_n = rest / slices;
  const int m0 = tile_m * S::rows, n0 = tile_n * S::cols;

  int Kc = g.Kc, nk_all;
  if constexpr (SEG) {
    nk_all = 0;
    for (int q = 0; q < sg.n; ++q) nk_all += sg.Kc[q] / S::step;  // whole steps (checked on the host)
  } else {
    nk_all = (Kc + S::step - 1) / S::step;
  }
  const int t_begin = slice * g.steps;
  const int t_end = t_begin + g.steps < nk_all ? t_begin + g.steps : nk_all;

  // ---- loads of 1 KiB
  const uint32_t ring0 = (uint32_t)(uintptr_t)TT_LDS_PTR(smem) + kTableBytes;
  constexpr int kChunks = 4 * KG;       // 16-byte chunks of a row of the activation stage
  constexpr int kRows = 64 / kChunks;   // rows of an instruction
  constexpr bool kHalfLoad = S::a_wave % 1024 != 0;  // the last of a wave's activation loads has half the lanes
  uint32_t a_off[S::a_loads], c_off, s_off;
  const int a_chunk_of_lane = lane % kChunks;
  auto row_swz = [&](int r) { return KG == 2 ? (r >> 1) & 7 : r & 15; };  // 16 rows of a chunk column fall on all banks
  auto swz = [&](int col) { return KG == 2 ? (col >> 3) & 1 : (col >> 2) & 3; };  // of a column's KG chunks of code bytes
  const int c_chunk = (lane % KG) ^ swz((64 / KG) * kg + lane / KG);
  auto set_offsets = [&](int kc) {
#pragma unroll
    for (int d = 0; d < S::a_loads; ++d) {
      const int r = wv * (S::rows / 8) + d * kRows + lane / kChunks;
      const int chunk = a_chunk_of_lane ^ row_swz(r);
      int row = m0 + r;
      row = row < g.M ? row : g.M - 1;
      a_off[d] = ((uint32_t)row * (uint32_t)kc + chunk * 8) * 2u;
    }
    int col = n0 + 64 * wn + (64 / KG) * kg + lane / KG;
    col = col < g.Nout ? col : g.Nout - 1;
    c_off = (uint32_t)(((int64_t)col * kc) >> 1) + 16 * c_chunk;
    if constexpr (MODE == 1) {
      int ob = (n0 >> 6) + wn;
      const int nob = g.Nout >> 6;
      ob = ob < nob ? ob : nob - 1;
      s_off = ((uint32_t)ob * (uint32_t)kc + 32 * kg + (lane & 31)) * 4u;
    } else {
      int sc = n0 + 64 * wn + lane;
      sc = sc < g.Nout ? sc : g.Nout - 1;
      s_off = MODE == 2 ? ((uint32_t)(kg >> 1) * (uint32_t)g.Nout + (uint32_t)sc) * 4u : ((uint32_t)sc * (uint32_t)(kc >> 6) + (uint32_t)(kg >> 1)) * 4u;
    }
  };
  const int64_t s_step = MODE == 1 ? S::step * 4 : MODE == 2 ? (int64_t)g.Nout * 4 * (KG / 2) : 4 * (KG / 2);
  // A contraction that is an odd number of 64 (KG 4): the last step starts 64 indices early and the waves of its first half,
  // whose indices the step before had, sit it out
  const int odd = KG == 4 && !SEG && (Kc & 64) != 0 ? 1 : 0;
  const char *pxb, *pcb, *psb;  // of the next step to be requested
  int sq = 0, sleft = 0;        // SEG: its segment, and that segment's steps from it on
  if constexpr (SEG) {
    int at = t_begin;
    while (at >= sg.Kc[sq] / S::step) at -= sg.Kc[sq++] / S::step;
    sleft = sg.Kc[sq] / S::step - at;
    set_offsets(sg.Kc[sq]);
    pxb = reinterpret_cast<const char*>(sg.X[sq]) + (int64_t)at * (S::step * 2);
    pcb = reinterpret_cast<const char*>(sg.codes[sq]) + (int64_t)at * (S::step / 2);
    psb = reinterpret_cast<const char*>(sg.scal[sq]) + (int64_t)at * (S::step * 4);
  } else {
    set_offsets(Kc);
    pxb = reinterpret_cast<const char*>(g.X) + (int64_t)t_begin * (S::step * 2);
    pcb = reinterpret_cast<const char*>(g.codes) + (int64_t)t_begin * (S::step / 2);
    psb = reinterpret_cast<const char*>(g.scal) + (int64_t)t_begin * s_step;
  }
  int requested = t_begin;  // the step the pointers stand at
  auto advance = [&]() {
    ++requested;
    if constexpr (SEG) {
      if (--sleft == 0 && sq + 1 < sg.n) {
        ++sq;
        sleft = sg.Kc[sq] / S::step;
        set_offsets(sg.Kc[sq]);
        pxb = reinterpret_cast<const char*>(sg.X[sq]);
        pcb = reinterpret_cast<const char*>(sg.codes[sq]);
        psb = reinterpret_cast<const char*>(sg.scal[sq]);
        return;
      }
    }
    pxb += S::step * 2;
    pcb += S::step / 2;
    psb += s_step;
    if constexpr (KG == 4 && !SEG) {
      if (odd && requested == nk_all - 1) {
        pxb -= 128;
        pcb -= 32;
        psb -= s_step / 2;
      }
    }
  };
  auto dma16 = [&](uint32_t voff, const char* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds) : "memory", "m0");
  };
  auto dma4 = [&](uint32_t voff, const char* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(base), "s"(lds) : "memory", "m0");
  };
  auto issue = [&](int stage, int d) {  // load d of the step the pointers stand at
    const uint32_t to = ring0 + stage * S::stage;
    if (d < S::a_loads) {
      if (!(kHalfLoad && d == S::a_loads - 1) || lane < 32) dma16(a_off[d], pxb, to + wv * S::a_wave + d * 1024);
    } else if (d == S::a_loads) dma16(c_off, pcb, to + S::a_bytes + (wn * KG + kg) * 1024);
    else dma4(s_off, psb, to + S::a_bytes + S::c_bytes + wv * 256);
  };

  if constexpr (KG == 4 && !SEG) {
    if (odd && t_begin == nk_all - 1) {  // a slice of this one step
      pxb -= 128;
      pcb -= 32;
      psb -= s_step / 2;
    }
  }
  // ---- the first steps' loads, then the table while they are under way
  const int n_steps = t_end - t_begin;
  const int filled = n_steps < S::stages ? n_steps : S::stages;
  for (int p = 0; p < filled; ++p) {
#pragma unroll
    for (int d = 0; d < S::loads; ++d) issue(p, d);
    advance();
  }
  {
    // (uniform indices: a vector load would wait for the loads above)
    float four[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) four[e] = round_to_bf16(kNF4Mid[(4 * wv + e) & 15]);
    const int of = lane >> 4;
    const float lo = of == 0 ? four[0] : of == 1 ? four[1] : of == 2 ? four[2] : four[3];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float hi = round_to_bf16(kNF4Mid[2 * r + (wv >> 2)]);
      *reinterpret_cast<f32x4_t*>(smem + (r * 512 + threadIdx.x) * 16) = f32x4_t{hi, lo, hi, lo};
    }
  }

  // ---- operands.  Lane (l31, h) holds the contraction indices 16 h + 8 ks .. + 7 of the wave's 32 for product ks of a step:
  //      two code dwords of its column, the chunks 2 h and 2 h + 1 of its row
  int x_at[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) x_at[ks] = l31 * (S::step * 2) + (((4 * kg + 2 * h + ks) ^ row_swz(l31)) << 4);
  auto read_x = [&](int stage, int ks, int i) {
    return *reinterpret_cast<const bf16x8_t*>(smem + kTableBytes + stage * S::stage + i * (32 * S::step * 2) + x_at[ks]);
  };
  const int c_at = S::a_bytes + wn * KG * 1024 + l31 * (16 * KG) + ((kg ^ swz(l31)) << 4) + 8 * h;
  auto read_codes = [&](int stage, int j) {
    return *reinterpret_cast<const u32x2_t*>(smem + kTableBytes + stage * S::stage + c_at + j * (512 * KG));
  };
  constexpr int kScalers = MODE == 1 ? 16 : 2;
  auto read_scalers = [&](int stage, float (&sc)[kScalers]) {
    const char* p = smem + kTableBytes + stage * S::stage + S::a_bytes + S::c_bytes + wv * 256;
    if constexpr (MODE == 1) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p + 64 * h + 16 * c);
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[4 * c + e] = a[e];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) sc[j] = *reinterpret_cast<const float*>(p + (32 * j + l31) * 4);
    }
  };
  const uint32_t lane8 = (lane & 31) * 8;
  auto fetch = [&](uint32_t code, int b) {  // the table lies at LDS address 0
    const uint32_t at = __builtin_amdgcn_perm(code, lane8, 0x0c0c0000u | (uint32_t)(4 + b) << 8);
    return *reinterpret_cast<const __attribute__((address_space(3))) f32x2_t*>(at);
  };
  auto finish = [&](const f32x2_t& p, const float (&sc)[kScalers], int q, int b) {
    if constexpr (MODE == 1) return pack_pair(p.x * sc[8 * (q >> 1) + 2 * b], p.y * sc[8 * (q >> 1) + 2 * b + 1]);
    else return pack_pair(p.x * sc[q & 1], p.y * sc[q & 1]);
  };

  f32x16_t acc[2][MT];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.f;
  // A step is four quarters of MT products each: column square j = q & 1, half ks = q >> 1 of the wave's contraction indices.
  // Beside quarter q the weights of quarter q + 1 are scaled and rounded and the table entries of quarter q + 2 requested;
  // those of quarters 0 and 1 of the next step beside quarters 2 and 3.
  bf16x8_t xf[2][MT];
  u32x4_t wf[4];
  f32x2_t pend[2][4];
  u32x2_t codes[2];
  float sc[kScalers];
  auto landed = [&](int left) {  // this wave's loads but those of the newest `left` steps, and everybody is here
    if (S::stages > 3 && left >= 3) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * S::loads) : "memory");
    else if (left >= 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * S::loads) : "memory");
    else if (left == 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(S::loads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  };
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the table's entries
  landed(filled - 1);
#pragma unroll
  for (int j = 0; j < 2; ++j) codes[j] = read_codes(0, j);
  read_scalers(0, sc);
#pragma unroll
  for (int i = 0; i < MT; ++i) xf[0][i] = read_x(0, 0, i);
#pragma unroll
  for (int b = 0; b < 4; ++b) pend[0][b] = fetch(codes[0].x, b);
#pragma unroll
  for (int b = 0; b < 4; ++b) pend[1][b] = fetch(codes[1].x, b);
#pragma unroll
  for (int i = 0; i < MT; ++i) xf[1][i] = read_x(0, 1, i);
#pragma unroll
  for (int b = 0; b < 4; ++b) wf[0][b] = finish(pend[0][b], sc, 0, b);

  int stage = 0;
  // The barrier of step t stands behind its first quarter: by then a wave has the step's operands in registers, so the loads of
  // step t + stages may take its stage, and everybody's loads of step t + 1 have landed.
  auto step = [&](int t, auto steady) {
    constexpr bool kSteady = decltype(steady)::value;
    const int old = stage;
    stage = stage == S::stages - 1 ? 0 : stage + 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q == 1) {
        // the four requests of quarter 0 are the youngest reads of LDS: the others, this step's operands among them, have arrived
        asm volatile("s_waitcnt lgkmcnt(4)" ::: "memory");
        if constexpr (kSteady) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S::stages - 2) * S::loads) : "memory");
        else landed(t_end - t - 2 < S::stages - 2 ? t_end - t - 2 : S::stages - 2);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        acc[q & 1][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wf[q]), xf[q >> 1][i], acc[q & 1][i], 0, 0, 0);
        if (q >= 2) xf[q - 2][i] = read_x(stage, q - 2, i);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int fin_at = q < 2 ? u * MT / 4 : q == 2 ? u * MT / 8 : MT / 2 + u * MT / 8;
          const int get_at = q == 0 ? u * MT / 4 + MT / 8 : q == 2 ? MT / 2 + u * MT / 8 : u * MT / 8;
          const int f = (q + 1) & 3, n = (q + 2) & 3;
          if (i == fin_at) wf[f][u] = finish(pend[f & 1][u], sc, f, u);
          if (i == get_at) pend[n & 1][u] = fetch(codes[n & 1][n >> 1], u);
        }
        if (q == 1 && i == MT / 2) {
#pragma unroll
          for (int j = 0; j < 2; ++j) codes[j] = read_codes(stage, j);
        }
        if (q == 2 && i == MT / 2) read_scalers(stage, sc);
#pragma unroll
        for (int d = 0; d < S::loads; ++d)
          if (kSteady && (q - 1) * MT + i == d * 2 * MT / S::loads) issue(old, d);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (kSteady) advance();
  };
  f32x16_t ended[FOLD ? 2 : 1][FOLD ? MT : 1];
  int left = FOLD ? g.chain : 0;
  auto fold = [&]() {
    if constexpr (FOLD) {
      if (--left > 0) return;
      left = g.chain;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            ended[j][i][v] += acc[j][i][v];
            acc[j][i][v] = 0.f;
          }
    }
  };
  if constexpr (FOLD) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) ended[j][i][v] = 0.f;
  }
  int t = t_begin;
  for (; t + S::stages < t_end; ++t) {
    step(t, std::true_type());
    fold();
  }
  const int t_stop = odd && kg < 2 && t_end == nk_all ? t_end - 1 : t_end;
  for (; t < t_stop; ++t) {
    step(t, std::false_type());
    fold();
  }
  if (t < t_end) asm volatile("s_barrier" ::: "memory");
  if constexpr (FOLD) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][i][v] += ended[j][i][v];
  }

  // ---- adapter: one product per 16 ranks, operands straight from global memory; lane (l31, h) holds ranks rc + 8 h .. + 7 of
  //      weight column / activation row l31 of its square.  The first ones are requested ahead of the exchange of the sums.
  constexpr int NJ = S::nj, MR = S::mr;
  const int mr0 = m0 + 32 * S::sq_i(kg, 0), nb = n0 + 64 * wn + 32 * S::sq_j(kg, 0);
  u32x4_t xraw[MR], wraw[NJ];
  auto adapter_rank = [&](int ad) {
    const bool none = (SEG ? sg.lX[ad] : g.lX) == nullptr || slice != 0;
    return none ? 0 : SEG ? sg.R[ad] : g.R;
  };
  auto request = [&](int ad, int rc) {
    const uint16_t* __restrict__ lX = SEG ? sg.lX[ad] : g.lX;
    const uint16_t* __restrict__ lW = SEG ? sg.lW[ad] : g.lW;
    const int R = SEG ? sg.R[ad] : g.R;
    const int r0 = rc + 8 * h;
    const bool in = r0 < R;  // R % 8 == 0: a lane's 8 indices are all in or all out
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      int row = mr0 + 32 * i + l31;
      row = row < g.M ? row : g.M - 1;
      xraw[i] = u32x4_t{0, 0, 0, 0};
      if (in) xraw[i] = *reinterpret_cast<const u32x4_t*>(lX + (int64_t)row * g.ldlx + r0);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      int col = nb + 32 * j + l31;
      col = col < g.Nout ? col : g.Nout - 1;
      wraw[j] = u32x4_t{0, 0, 0, 0};
      if (in) {
        if (g.lw_row_major) {
          wraw[j] = *reinterpret_cast<const u32x4_t*>(lW + (int64_t)col * R + r0);
        } else {
          uint32_t e[8];
#pragma unroll
          for (int d = 0; d < 8; ++d) e[d] = lW[(int64_t)(r0 + d) * g.Nout + col];
#pragma unroll
          for (int d = 0; d < 4; ++d) wraw[j][d] = e[2 * d] | (e[2 * d + 1] << 16);
        }
      }
    }
  };
  if (adapter_rank(0) > 0) request(0, 0);

  // ---- the wave groups' sums, each square's to the group that finishes it: (s0 + s1) + (s2 + s3) whoever adds them
  f32x16_t res[NJ][MR];
  __syncthreads();
  auto slot = [&](int dst, int e, int v4, int other) {  // other: source ^ dst, 1 .. KG - 1
    return smem + ((((dst * S::wn + wn) * (KG - 1) + other - 1) * S::own + e) * 4 + v4) * 1024 + lane * 16;
  };
#pragma unroll
  for (int k = 0; k < KG; ++k) {
    if (kg == k) {
#pragma unroll
      for (int d = 0; d < KG; ++d)
#pragma unroll
        for (int e = 0; e < S::own; ++e) {
          const f32x16_t a = acc[S::sq_j(d, e)][S::sq_i(d, e)];
          if (d == k) {
            res[NJ == 2 ? e & 1 : 0][NJ == 2 ? e >> 1 : e] = a;
          } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) *reinterpret_cast<f32x4_t*>(slot(d, e, v, d ^ k)) = f32x4_t{a[4 * v], a[4 * v + 1], a[4 * v + 2], a[4 * v + 3]};
          }
        }
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < S::own; ++e)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      f32x16_t& r = res[NJ == 2 ? e & 1 : 0][NJ == 2 ? e >> 1 : e];
      const f32x4_t o = *reinterpret_cast<const f32x4_t*>(slot(kg, e, v, 1));
#pragma unroll
      for (int w = 0; w < 4; ++w) r[4 * v + w] += o[w];
      if constexpr (KG == 4) {
        const f32x4_t p = *reinterpret_cast<const f32x4_t*>(slot(kg, e, v, 2)) + *reinterpret_cast<const f32x4_t*>(slot(kg, e, v, 3));
#pragma unroll
        for (int w = 0; w < 4; ++w) r[4 * v + w] += p[w];
      }
    }

  const int n_adapters = SEG ? sg.n : 1;
  for (int ad = 0; ad < n_adapters; ++ad) {
    const int R = adapter_rank(ad);
    for (int rc = 0; rc < R; rc += 16) {
      if (ad > 0 || rc > 0) request(ad, rc);
#pragma unroll
      for (int i = 0; i < MR; ++i) {
        u32x4_t raw = xraw[i];
        if (g.lscale != 1.0f) {
#pragma unroll
          for (int d = 0; d < 4; ++d) raw[d] = pack_pair(bits_f32(raw[d] << 16) * g.lscale, bits_f32(raw[d] & 0xffff0000u) * g.lscale);
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          res[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wraw[j]), __builtin_bit_cast(bf16x8_t, raw), res[j][i], 0, 0, 0);
      }
    }
  }

  // ---- res[j][i][v] = C[mr0 + 32 i + l31][nb + 32 j + 8 (v / 4) + 4 h + v % 4]
  if (nb >= g.Nout) return;  // the wave's columns lie outside (no barrier follows)
  if (split) {
    float* P = g.part + (int64_t)slice * g.M * g.Nout + nb + 4 * h;
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      const int row = mr0 + 32 * i + l31;
      if (row >= g.M) continue;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          *reinterpret_cast<f32x4_t*>(P + (int64_t)row * g.Nout + 32 * j + 8 * v) =
              f32x4_t{res[j][i][4 * v], res[j][i][4 * v + 1], res[j][i][4 * v + 2], res[j][i][4 * v + 3]};
    }
    return;
  }
  // rows of 64 NJ bytes through LDS (a region that only this wave has read), chunk c of row r in slot c ^ (r % (4 NJ))
  constexpr int kBand = 64 * NJ, kSlots = 4 * NJ;
  char* mine = smem + (kg * S::wn + wn) * (KG - 1) * S::own * 4096;
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float b4[4] = {0.f, 0.f, 0.f, 0.f}, c4[4] = {1.f, 1.f, 1.f, 1.f};
      if (g.bias) {
        const u32x2_t bb = *reinterpret_cast<const u32x2_t*>(g.bias + nb + 32 * j + 8 * v + 4 * h);
        b4[0] = bits_f32(bb.x << 16); b4[1] = bits_f32(bb.x & 0xffff0000u);
        b4[2] = bits_f32(bb.y << 16); b4[3] = bits_f32(bb.y & 0xffff0000u);
      }
      if (g.cscale) {
        const u32x2_t cc = *reinterpret_cast<const u32x2_t*>(g.cscale + nb + 32 * j + 8 * v + 4 * h);
        c4[0] = bits_f32(cc.x << 16); c4[1] = bits_f32(cc.x & 0xffff0000u);
        c4[2] = bits_f32(cc.y << 16); c4[3] = bits_f32(cc.y & 0xffff0000u);
      }
#pragma unroll
      for (int i = 0; i < MR; ++i) {
        const int r = 32 * i + l31;
        u32x2_t o;
        o.x = pack_pair((res[j][i][4 * v] + b4[0]) * c4[0], (res[j][i][4 * v + 1] + b4[1]) * c4[1]);
        o.y = pack_pair((res[j][i][4 * v + 2] + b4[2]) * c4[2], (res[j][i][4 * v + 3] + b4[3]) * c4[3]);
        *reinterpret_cast<u32x2_t*>(mine + r * kBand + (((4 * j + v) ^ (r & (kSlots - 1))) << 4) + 8 * h) = o;
      }
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int c = lane % kSlots;
  uint16_t* crow = g.C + nb + 8 * c;
#pragma unroll
  for (int p = 0; p < 32 * MR * kSlots / 64; ++p) {
    const int r = (64 / kSlots) * p + lane / kSlots;
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(mine + r * kBand + ((c ^ (r & (kSlots - 1))) << 4));
    if (mr0 + r < g.M) *reinterpret_cast<u32x4_t*>(crow + (int64_t)(mr0 + r) * g.Nout) = v;
  }
#endif
}

template <int MT, int KG, int MODE, int FORM, bool FOLD>
int launch(RsArgs& g, const std::conditional_t<FORM == kMembers, RsMembers, RsSegs>& sg, hipStream_t s) {
  using S = NMid<MT, KG>;
  auto* fn = &nf4_gemm_mid_kernel<MT, KG, MODE, FORM, FOLD>;
  static bool set[64] = {};  // the LDS limit is a per-device attribute of the function (a race only repeats the call)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (dev < 0 || !set[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, S::lds);
    if (e != hipSuccess) return fail(TTAMD_ELAUNCH, "nf4_gemm_mid: cannot reserve %d bytes of LDS: %s", S::lds, hipGetErrorString(e));
    if (dev >= 0) set[dev] = true;
  }
  g.tiles_m = (g.M + S::rows - 1) / S::rows;
  g.tiles_n = (g.Nout + S::cols - 1) / S::cols;
  g.items = g.tiles_m * g.tiles_n * g.slices;
  g.per_xcd = (g.items + 7) / 8;
  if constexpr (FORM == kMembers) g.per_xcd = sg.slot_end[sg.n - 1];
  fn<<<dim3(8u * g.per_xcd), dim3(512), S::lds, s>>>(g, sg);
  return check_launch("nf4_gemm_mid");
}

template <int MODE, int FORM>
int launch_rows(RsArgs& g, int rows, bool fold, const std::conditional_t<FORM == kMembers, RsMembers, RsSegs>& sg, hipStream_t s) {
  if (rows == 128) return launch<4, 2, MODE, FORM, false>(g, sg, s);
  if (rows == 96) return launch<3, 2, MODE, FORM, false>(g, sg, s);
  return fold ? launch<2, 4, MODE, FORM, true>(g, sg, s) : launch<2, 4, MODE, FORM, false>(g, sg, s);
}

// Slices of a contraction on tiles of 128 x 256, for launches of half a round of them to a whole one: costs in us of a round 64 at
// 4096 steps, the slabs' way out and back at 4 TB/s, the sum's launch 6; a fuller chip clocks lower, so a sixth has to be gained.
int part_filled_chains(int64_t tiles, int64_t M, int64_t Nout, int64_t Kc) {
  const double whole = 64.0 * (double)Kc / 4096.0;
  double best = whole / 1.2;
  int best_sp = 1;
  for (int sp = 2; sp <= 8 && Kc / sp >= 1024; ++sp) {
    const double cost = whole * (double)((tiles * sp + 255) / 256) / sp + 6.0 + (double)sp * (double)(M * Nout) * 8.0 / 4e6;
    if (cost < best) {
      best = cost;
      best_sp = sp;
    }
  }
  return best_sp;
}

}  // namespace

int nmid_cols(int rows) { return rows == 64 ? 128 : 256; }

// How many chains of fp32 sums an output's contraction is cut into at least: as many as slices of it, on tiles of 128 x 256, would
// fill the chip about once (at least 256 indices each, at most 16).  More only shorten a chain; fewer would lengthen it.
int nmid_min_chains(int64_t M, int64_t Nout, int64_t Kc) {
  const int64_t tiles = ((M + 127) / 128) * ((Nout + 255) / 256);
  if (tiles > 128) return tiles < 256 && !dense_path_applies(M, Nout, Kc) ? part_filled_chains(tiles, M, Nout, Kc) : 1;
  if (tiles > 64 && Kc < 4096) return 1;
  int64_t sp = 256 / tiles;
  const int64_t by_k = (Kc / 64) / 4;
  sp = sp < by_k ? sp : by_k;
  sp = sp < 16 ? sp : 16;
  return sp < 2 ? 1 : (int)sp;
}

namespace {
// The time in us of a launch: a start, a term for each round of 256 workgroups and each of its steps, one for the steps weighed by
// how full their round is (the clock falls with the load), and for slices the sum's launch and the slabs.  The terms are fitted
// to 8300 launches (24 weights of 256 x 1024 to 14336 x 4096, 33 - 2047 rows, forward and grad-input); the pick by them is 0.3 %
// slower than the fastest on average.
struct NMidTerms {
  int rows;
  double start, round, step, full_step, sum, slab;
};
constexpr NMidTerms kTerms[] = {{64, 4.08, 2.90, 0.521, 0.156, 2.18, 2.08}, {96, 4.95, 4.08, 0.557, 0.227, 2.86, 1.25}, {128, 4.39, 5.21, 0.589, 0.326, 3.06, 1.13}};

double launch_cost(const NMidTerms& c, int64_t items, int64_t steps, int64_t slabs, double elements) {
  const int64_t full = items / 256, rounds = (items + 255) / 256;
  const double part = (double)(items % 256) / 256;
  const double t = c.start + rounds * (c.round + c.step * (double)steps) + c.full_step * ((double)full + part * part) * (double)steps;
  return slabs > 1 ? t + c.sum + c.slab * 1e-6 * (double)slabs * elements : t;
}
int64_t tiles_of(int rows, int64_t M, int64_t Nout) { return ((M + rows - 1) / rows) * ((Nout + nmid_cols(rows) - 1) / nmid_cols(rows)); }
}  // namespace

// Wide forwards (a gate or up projection: outputs twice the contraction and more) whose pair fills half the chip with whole
// contractions stay whole.  Slices gain one of them 4 % mostly and up to 17 (nine widths at 150 - 800 tokens, us: 8192 x 3072 at 260 36.6 ->
// 32.6, 9728 x 3584 at 200 41.8 -> 34.8, at 384 44.7 -> 46.5) and cost the pair's one launch, whose members keep their own slices,
// 14 - 60 % (42.1 -> 64.7, 47.1 -> 67.9, 6912 x 2560 at 384 40.0 -> 64.0).
//
// The query and the call plan anew, and a pass of small layers waits for the host: the search ends where the slabs alone cost more
// than the best plan so far (0.05 - 0.2 us; all 48 plans took 0.2 - 0.4).
NMidPlan nmid_plan(int64_t M, int64_t Nout, int64_t Kc, bool may_slice, bool by_128, bool forward, double* cost) {
  const int chains = nmid_min_chains(M, Nout, Kc);
  const bool sliceable = may_slice && !(chains == 1 && forward && Nout >= 2 * Kc && tiles_of(128, M, Nout) > 64);
  const double elements = (double)M * (double)Nout;
  const int most = sliceable ? (int)(Kc / 256 < 16 ? Kc / 256 : 16) : 1;
  NMidPlan p = {};
  *cost = 0;
  for (const auto& c : kTerms) {
    const int groups = c.rows == 64 ? 4 : 2, step = 32 * groups;
    if (c.rows == 64 && (!by_128 || Kc < 128)) continue;
    const int64_t nk = (Kc + step - 1) / step, tiles = tiles_of(c.rows, M, Nout);
    const double least = c.start + c.round + c.step * (double)tiles * (double)nk / 256 + c.sum;  // of slices, but for the slabs
    for (int n = 1; n == 1 || n <= most; ++n) {
      if (n > 1 && p.rows != 0 && least + c.slab * 1e-6 * (double)n * elements > *cost) break;
      // the wave groups' sums are chains of their own; whole contractions on the smallest tiles can end theirs early (no slower
      // beyond 1 - 2 %), the others have no registers for it
      const bool fold = n * groups < chains;
      if (fold && may_slice && (c.rows != 64 || n > 1)) continue;
      const int64_t steps = (nk + n - 1) / n;
      if (n > 1 && (nk + steps - 1) / steps != n) continue;
      const double t = launch_cost(c, tiles * n, steps, n, elements);
      if (p.rows == 0 || t < *cost) {
        *cost = t;
        p.rows = c.rows;
        p.slices = n;
        p.steps = (int)steps;
        p.chain = fold && c.rows == 64 ? 2 * (int)((Kc / 64 + chains - 1) / chains) : 0;
      }
    }
  }
  return p;
}

int nmid_group_rows(int64_t M, const int64_t* Nout, const NMidPlan* p, int n) {
  if (p[0].rows == 64) return 64;
  int best = 0;
  double least = 0;
  for (const auto& c : kTerms) {
    if (c.rows == 64) continue;
    int64_t items = 0;
    double steps = 0;  // of a workgroup, on average
    for (int i = 0; i < n; ++i) {
      const int64_t k = tiles_of(c.rows, M, Nout[i]) * (int64_t)p[i].slices;
      items += k;
      steps += (double)k * (double)p[i].steps;
    }
    const double t = launch_cost(c, items, (int64_t)(steps / (double)items), 1, 0);
    if (best == 0 || t < least) {
      least = t;
      best = c.rows;
    }
  }
  return best;
}

int run_nf4_gemm_mid(int mode, RsArgs& g, const NMidPlan& p, const RsSegs* segs, const RsMembers* members, hipStream_t s) {
  g.slices = p.slices;
  g.steps = p.steps;
  g.chain = p.chain;
  if (members) return launch_rows<2, kMembers>(g, p.rows, p.chain > 0, *members, s);
  if (segs) return launch_rows<1, kSegments>(g, p.rows, p.chain > 0, *segs, s);
  static const RsSegs none = {};
  return mode == 1   ? launch_rows<1, kPlain>(g, p.rows, p.chain > 0, none, s)
         : mode == 2 ? launch_rows<2, kPlain>(g, p.rows, p.chain > 0, none, s)
                     : launch_rows<0, kPlain>(g, p.rows, p.chain > 0, none, s);
}

}  // namespace ttamd
