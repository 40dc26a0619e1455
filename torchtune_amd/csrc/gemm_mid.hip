// Plain bf16 products of a few dozen to some thousand rows: the three matmuls of a fake-quantised linear below the sizes of the
// 256 x 256-tile kernels (torchtune/modules: F.linear(fq(x), fq(W)) and what autograd derives from it).
//
//   kind 0   C[M, N] = A[M, K] . B[N, K]^T (+ bias)     forward
//   kind 1   C[M, N] = A[M, K] . B[K, N]                grad-input
//   kind 2   C[M, N] = A[K, M]^T . B[K, N]              weight gradient (the contraction runs over the tokens)
//
// gemm_mid_kernel (kinds 0 and 1): eight waves per tile of 64, 128 or 256 rows and 128 columns.  A step is 64 contraction
// indices; four waves (2 x 2, half the rows and columns each) multiply its first 32, the other four its second 32, and the two
// sums are added through LDS at the end.  So a tile keeps two waves on every SIMD, a barrier comes once per 64 indices, and
// what lies along the contraction is fetched in whole lines of 128 bytes: with steps of 32 a line was fetched twice (1024 x
// 8192 x 2048, kind 0: 7.7 million L2 requests, 4.2 with whole lines), which is what bound the forward products.
//   The tile's height trades LDS and L2 traffic (per step 512, 768 and 1152 cycles of LDS against 256, 512 and 1024 of the
// matrix pipes) for workgroups: 256 rows where they fill the CUs (1000 x 8192 x 2048 44.4 -> 33.3 us, of which the matrix
// pipes take 21 at the 1.6 GHz that the card holds under them), 128 below (1000 x 2048 x 8192 in two slices 50.8 -> 41.7),
// 64 where the chip would be half idle (1000 x 2048 x 2048 21.1 -> 15.1).  The 64-row tile takes half a CU's LDS: two run there.
// gemm_mid_pair_kernel (kind 2, and kind 1 over a short contraction of many tiles): four waves per tile of 128 x 128, two
// workgroups per CU, steps of 32.  Both operands of kind 2 lie across the contraction, in lines of 256 bytes, and its
// contraction (the tokens) is short: two independent workgroups hide each other's first loads and last stores (8192 x 2048
// outputs over 1000 tokens 52.6 us, on tiles as gemm_mid_kernel's 55 - 65).  Weight gradients of more outputs run on the
// 256 x 256 tiles of gemm_tn.hip (31.3 us there).
// Launches of few tiles cut the contraction into slices (fp32 slabs, added in slice order by gemm_mid_reduce_kernel).
// Over 380 products of kinds 0 and 1 (40 - 8192 rows, 256 - 14336 columns) these two take 0.84 of the time of the four-wave
// kernel alone; where both cut the contraction alike the sums are closer to the exact ones (2.7e-7 against 3.9e-7 over 8192
// indices in two slices): two chains of half the length.  A training pass of a 1B-shaped layer over 1000 tokens with its 21 products: 825 -> 735 us, with the wide
// tiles for its weight gradients 714 (host-bound there).
#include "common.h"
#include "group.h"
#include "nf4_math.h"

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

struct MidArgs {
  const uint16_t* A;
  const uint16_t* B;
  const uint16_t* bias;  // [N] or null
  uint16_t* C;
  float* part;           // SPLIT: [slices, M, N]
  int M, N, K;
  int tiles_m, tiles, per_xcd;
  int slices, steps_per_slice;
  int chain;             // FOLD: steps of a chain, even
};

constexpr int kMidCols = 128;  // columns of a tile
constexpr int kMidStep = 64;   // contraction indices of a step

// MT: groups of 16 rows per wave, so a tile has 32 MT; WGS: workgroups per CU
template <int MT, int WGS>
struct MidShape {
  static constexpr int rows = 32 * MT;
  static constexpr int a_bytes = rows * kMidStep * 2;
  static constexpr int b_bytes = kMidCols * kMidStep * 2;
  static constexpr int stage = a_bytes + b_bytes;
  static constexpr int stages = 160 * 1024 / WGS / stage;  // 3, 5 and 3 for 64, 128 and 256 rows
  static constexpr int lds = stages * stage;
  static constexpr int a_loads = MT / 2, b_loads = 2, loads = a_loads + b_loads;  // per wave and step, 1 KiB each
};

// FOLD: the chains end after g.chain steps and are added up in registers (not with 256 rows: they fill the registers).
template <bool B_COL, bool SPLIT, int MT, int WGS, bool FOLD>
__global__ __launch_bounds__(512, 2 * WGS) void gemm_mid_kernel(const MidArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  using S = MidShape<MT, WGS>;
  static_assert(S::stages >= 3, "a step in registers, one landed, one in flight");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // workgroup ids go round-robin to the 8 XCDs: each gets a run of neighbouring tiles, row tiles first, with all their slices
  // (an equal share of the items: dealt out slice by slice, 84 tiles in 3 slices put 33 on some XCDs' 32 CUs)
  const int item = (int)(blockIdx.x & 7) * g.per_xcd + (int)(blockIdx.x >> 3);
  const int tile = SPLIT ? item / g.slices : item, slice = SPLIT ? item - tile * g.slices : 0;
  if ((int)(blockIdx.x >> 3) >= g.per_xcd || tile >= g.tiles) return;
  const int m0 = (tile % g.tiles_m) * S::rows, n0 = (tile / g.tiles_m) * kMidCols;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wv >> 2, wm = (wv >> 1) & 1, wn = wv & 1;
  const int l15 = lane & 15, g4 = lane >> 4;
  const int nk_all = g.K / kMidStep;
  const int t_begin = SPLIT ? slice * g.steps_per_slice : 0;
  const int t_end = SPLIT ? (t_begin + g.steps_per_slice < nk_all ? t_begin + g.steps_per_slice : nk_all) : nk_all;
  const uint32_t lds0 = (uint32_t)(uintptr_t)TT_LDS_PTR(smem);

  // ---- loads of 1 KiB.  Along the contraction: 8 rows of 128 bytes; 16-byte chunk c of row r in slot c ^ (r % 8).
  //      Across it: 4 contraction indices of 256 bytes (128 columns); chunk c of index r in slot c ^ 2 (r % 4) ^ 8 ((r / 8) % 2).
  //      Rows and columns beyond the matrix repeat a valid one (never stored); K is a whole number of steps.
  uint32_t voff[S::loads];
  auto offset = [&](bool col, int q, int first, int extent, int ld) {
    if (col) {
      const int r = 4 * q + (lane >> 4);
      const int c = first + 8 * ((lane & 15) ^ ((r & 3) << 1) ^ (((r >> 3) & 1) << 3));
      return (uint32_t)((int64_t)r * ld + (c < extent ? c : first)) * 2u;
    }
    const int row = first + 8 * q + (lane >> 3);
    return (uint32_t)((int64_t)(row < extent ? row : extent - 1) * ld * 2 + (((lane & 7) ^ (lane >> 3)) << 4));
  };
  const int ldb = B_COL ? g.N : g.K;
#pragma unroll
  for (int d = 0; d < S::loads; ++d)
    voff[d] = d < S::a_loads ? offset(false, wv * S::a_loads + d, m0, g.M, g.K) : offset(B_COL, wv * S::b_loads + d - S::a_loads, n0, g.N, ldb);
  const int64_t a_step = kMidStep * 2, b_step = B_COL ? (int64_t)ldb * kMidStep * 2 : kMidStep * 2;
  auto issue = [&](int t, int stage, int d) {
    const bool a = d < S::a_loads;
    const int q = a ? wv * S::a_loads + d : wv * S::b_loads + d - S::a_loads;
    const char* base = a ? reinterpret_cast<const char*>(g.A) + (int64_t)t * a_step : reinterpret_cast<const char*>(g.B) + (int64_t)t * b_step;
    const uint32_t to = lds0 + stage * S::stage + (a ? 0 : S::a_bytes) + q * 1024;
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff[d]), "s"(base), "s"(to) : "memory", "m0");
  };

  // ---- operand reads: fragment e (16 rows / columns) of the wave's half of the contraction step
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  const int row_at = l15 * 128 + (((4 * kg + g4) ^ (l15 & 7)) << 4);
  int col_at[4];  // lane (l15, g4) points at contraction index 8 g4 + l15 / 4 (+ 4), columns 4 (l15 % 4) .. + 3 of group e
#pragma unroll
  for (int e = 0; e < 4; ++e) col_at[e] = 8192 * kg + (8 * g4 + (l15 >> 2)) * 256 + 8 * (l15 & 3) + 32 * (e ^ (l15 >> 2));
  auto fragment = [&](bool col, const char* base, int group) {
    if (col) {
      const char* p = base + col_at[group & 3] + 128 * ((group >> 2) ^ (g4 & 1));
      const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p));
      const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p + 1024));
      typedef short s16x8_t __attribute__((ext_vector_type(8)));
      const s16x8_t both = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      return __builtin_bit_cast(bf16x8_t, both);
    }
    return *reinterpret_cast<const bf16x8_t*>(base + row_at + 2048 * group);
  };
  auto read_a = [&](int stage, int i) { return fragment(false, smem + stage * S::stage, MT * wm + i); };
  auto read_b = [&](int stage, int j) { return fragment(B_COL, smem + stage * S::stage + S::a_bytes, 4 * wn + j); };

  f32x4_t acc[4][MT];  // [n tile][m tile]
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // While step t is multiplied from registers, the operands of step t + 1 replace them: row group i as soon as it is multiplied.
  // The barrier at the head of step t: a wave's loads of step t + 1 are the oldest in flight, so after it everybody's have
  // landed; and everybody's reads of step t are complete (lgkmcnt), so the loads of step t + stages may take its stage.  They
  // go out one between the row groups: in front of the products the waves would queue for the address unit.
  bf16x8_t af[MT], bf[2][4];
  const int filled = t_end - t_begin < S::stages ? t_end - t_begin : S::stages;
  for (int p = 0; p < filled; ++p) {
#pragma unroll
    for (int d = 0; d < S::loads; ++d) issue(t_begin + p, p, d);
  }
  // every wave's loads but those of the newest `left` steps have landed
  auto landed = [&](int left) {
    if (left >= 4) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(4 * S::loads) : "memory");
    else if (left == 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(3 * S::loads) : "memory");
    else if (left == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * S::loads) : "memory");
    else if (left == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S::loads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  static_assert(S::stages <= 5, "landed() tells four steps apart");
  landed(filled - 1);
#pragma unroll
  for (int e = 0; e < MT; ++e) af[e] = read_a(0, e);
#pragma unroll
  for (int e = 0; e < 4; ++e) bf[0][e] = read_b(0, e);
  int stage = 0;  // of step t
  auto step = [&](int t, int set, auto steady) {
    if constexpr (decltype(steady)::value) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S::stages - 2) * S::loads) : "memory");
    else landed(t_end - t - 2 < S::stages - 2 ? t_end - t - 2 : S::stages - 2);
    const int old = stage;
    stage = stage == S::stages - 1 ? 0 : stage + 1;
    const bool more = decltype(steady)::value || t + S::stages < t_end;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[set][j], af[i], acc[j][i], 0, 0, 0);
      af[i] = read_a(stage, i);
      constexpr int per = MT >= 4 ? 1 : 4 / MT;
#pragma unroll
      for (int e = per * i; e < per * (i + 1) && e < 4; ++e) bf[set ^ 1][e] = read_b(stage, e);
      constexpr int lper = (S::loads + MT - 1) / MT;
#pragma unroll
      for (int d = lper * i; d < lper * (i + 1) && d < S::loads; ++d)
        if (more) issue(t + S::stages, old, d);
    }
  };
  f32x4_t ended[FOLD ? 4 : 1][MT];  // the chains that have ended
  int left = FOLD ? g.chain : 0;    // steps of the present one
  auto fold = [&](bool last) {
    if constexpr (FOLD) {
      left -= 2;
      if (left > 0 && !last) return;
      left = g.chain;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          ended[j][i] += acc[j][i];
          acc[j][i] = last ? ended[j][i] : f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
  };
#pragma unroll
  for (int j = 0; j < (FOLD ? 4 : 1); ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) ended[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int t = t_begin;
  for (; t + 1 + S::stages < t_end; t += 2) {
    step(t, 0, std::true_type());
    step(t + 1, 1, std::true_type());
    fold(false);
  }
  for (; t < t_end; t += 2) {
    step(t, 0, std::false_type());
    if (t + 1 < t_end) step(t + 1, 1, std::false_type());
    fold(t + 2 >= t_end);
  }

  // ---- the two halves of each step's contraction: a wave keeps the columns 32 kg .. + 31 of its 64 and hands over the rest
  __syncthreads();  // every wave has read its last step: the ring is free
  f32x4_t sum[2][MT];
  auto hand_over = [&](const f32x4_t(&give)[MT], int j) {
#pragma unroll
    for (int i = 0; i < MT; ++i) *reinterpret_cast<f32x4_t*>(smem + ((wv * 2 + j) * MT + i) * 1024 + lane * 16) = give[i];
  };
  auto take = [&](const f32x4_t(&keep)[MT], int j) {
#pragma unroll
    for (int i = 0; i < MT; ++i) sum[j][i] = keep[i] + *reinterpret_cast<const f32x4_t*>(smem + (((wv ^ 4) * 2 + j) * MT + i) * 1024 + lane * 16);
  };
  if (kg == 0) { hand_over(acc[2], 0); hand_over(acc[3], 1); }
  else { hand_over(acc[0], 0); hand_over(acc[1], 1); }
  __syncthreads();
  if (kg == 0) { take(acc[0], 0); take(acc[1], 1); }
  else { take(acc[2], 0); take(acc[3], 1); }

  // sum[j][i][v] = C[m0 + 16 MT wm + 16 i + l15][n0 + 64 wn + 32 kg + 16 j + 4 g4 + v]
  const int nb = n0 + 64 * wn + 32 * kg;
  if constexpr (SPLIT) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = m0 + 16 * (MT * wm + i) + l15;
      if (m >= g.M) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = nb + 16 * j + 4 * g4;
        if (n < g.N) *reinterpret_cast<f32x4_t*>(g.part + ((int64_t)slice * g.M + m) * g.N + n) = sum[j][i];
      }
    }
  } else {
    __syncthreads();  // everybody has read its halves
    // the tile in bf16: rows of 256 bytes, chunk c of row r in slot c ^ (r % 16)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float b4[4] = {0.f, 0.f, 0.f, 0.f};
      if (g.bias && nb + 16 * j < g.N) {
        const u32x2_t b = *reinterpret_cast<const u32x2_t*>(g.bias + nb + 16 * j + 4 * g4);
        b4[0] = lo_of(b.x); b4[1] = hi_of(b.x); b4[2] = lo_of(b.y); b4[3] = hi_of(b.y);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        u32x2_t o;
        o.x = pack_pair(sum[j][i][0] + b4[0], sum[j][i][1] + b4[1]);
        o.y = pack_pair(sum[j][i][2] + b4[2], sum[j][i][3] + b4[3]);
        const int chunk = 8 * wn + 4 * kg + 2 * j + (g4 >> 1);
        *reinterpret_cast<u32x2_t*>(smem + (16 * (MT * wm + i) + l15) * 256 + ((chunk ^ l15) << 4) + 8 * (g4 & 1)) = o;
      }
    }
    __syncthreads();
    const int c = threadIdx.x & 15;
    if (n0 + 8 * c < g.N) {  // N % 8 == 0
#pragma unroll
      for (int p = 0; p < MT; ++p) {
        const int r = 32 * p + (threadIdx.x >> 4);
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(smem + r * 256 + ((c ^ (r & 15)) << 4));
        if (m0 + r < g.M) *reinterpret_cast<u32x4_t*>(g.C + (int64_t)(m0 + r) * g.N + n0 + 8 * c) = v;
      }
    }
  }
#endif
}

// ---------------------------------------------------------------------------------------------------
constexpr int kPairTile = 128;
constexpr int kPairOperand = 8192;              // 128 x 32 bf16
constexpr int kPairStage = 2 * kPairOperand;
constexpr int kPairStages = 5;
constexpr int kPairLds = kPairStages * kPairStage;

__device__ __constant__ u32x4_t kMidZero = {0, 0, 0, 0};

template <bool A_COL, bool SPLIT>
__global__ __launch_bounds__(256, 2) void gemm_mid_pair_kernel(const MidArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // workgroup ids go round-robin to the 8 XCDs: each gets a run of neighbouring tiles, row tiles first
  const int tile = (int)(blockIdx.x & 7) * g.per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= g.per_xcd || tile >= g.tiles) return;
  const int m0 = (tile % g.tiles_m) * kPairTile, n0 = (tile / g.tiles_m) * kPairTile;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv >> 1, wn = wv & 1;
  const int l15 = lane & 15, g4 = lane >> 4;
  const int nk_all = (g.K + 31) >> 5;
  const int t_begin = SPLIT ? (int)blockIdx.y * g.steps_per_slice : 0;
  const int t_end = SPLIT ? (t_begin + g.steps_per_slice < nk_all ? t_begin + g.steps_per_slice : nk_all) : nk_all;
  const uint32_t lds0 = (uint32_t)(uintptr_t)TT_LDS_PTR(smem);

  // ---- loads: two instructions of 1 KiB per wave, operand and step.
  //      Along the contraction: rows 32 wv + 16 d + lane / 4 of 64 bytes; 16-byte chunk c of row r in slot c ^ -(r / 4) % 4 (the
  //      negation because a 16-byte read serves rows 0 - 3, 12 - 15 of one chunk column together with 4 - 11 of the next).
  //      Across it: contraction indices 8 wv + 4 d + lane / 16, 256 bytes of the tile's 128 columns each; chunk c of index r in
  //      slot c ^ 2 (r % 4) ^ 8 ((r / 8) % 2).
  //      Rows and columns beyond the matrix repeat a valid one (never stored); contraction indices beyond K are zeros.
  uint32_t voff[2][2];  // [operand][d]
  int krow[2];          // across: the lane's contraction index within a step
  auto offsets = [&](int op, bool col, int first, int extent, int ld) {
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      if (col) {
        const int r = 8 * wv + 4 * d + (lane >> 4);
        const int chunk = (lane & 15) ^ ((r & 3) << 1) ^ (((r >> 3) & 1) << 3);
        const int c = first + 8 * chunk < extent ? first + 8 * chunk : first;
        voff[op][d] = (uint32_t)((int64_t)r * ld + c) * 2u;
        krow[d] = r;
      } else {
        const int r = 32 * wv + 16 * d + (lane >> 2);
        const int chunk = (lane & 3) ^ (-(lane >> 4) & 3);
        const int row = first + r < extent ? first + r : extent - 1;
        voff[op][d] = (uint32_t)((int64_t)row * ld * 2 + chunk * 16);
      }
    }
  };
  const int lda = A_COL ? g.M : g.K, ldb = g.N;
  offsets(0, A_COL, m0, g.M, lda);
  offsets(1, true, n0, g.N, ldb);
  const int64_t a_step = A_COL ? (int64_t)lda * 64 : 64, b_step = (int64_t)ldb * 64;
  const bool ragged = (g.K & 31) != 0;  // only across the contraction on both sides (checked on the host)
  auto issue = [&](int t, int stage) {
    const int tk = t < t_end ? t : t_end - 1;  // past the end: the last step again (the waits count a fixed number in flight)
    const char* ab = reinterpret_cast<const char*>(g.A) + (int64_t)tk * a_step;
    const char* bb = reinterpret_cast<const char*>(g.B) + (int64_t)tk * b_step;
    const uint32_t sa = lds0 + stage * kPairStage + wv * 2048;
    if (A_COL && ragged && tk == nk_all - 1) {
      const char* z = reinterpret_cast<const char*>(&kMidZero);
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const bool in = 32 * tk + krow[d] < g.K;
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(in ? ab + voff[0][d] : z), "s"(sa + 1024u * d) : "memory", "m0");
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(in ? bb + voff[1][d] : z), "s"(sa + kPairOperand + 1024u * d) : "memory", "m0");
      }
      return;
    }
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff[0][d]), "s"(ab), "s"(sa + 1024u * d) : "memory", "m0");
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff[1][d]), "s"(bb), "s"(sa + kPairOperand + 1024u * d) : "memory", "m0");
    }
  };

  // ---- operand reads: fragment e (16 rows / columns) of a wave's four
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  const int row_at = l15 * 64 + ((g4 ^ (-(l15 >> 2) & 3)) << 4);
  int col_at[4];  // lane (l15, g4) points at contraction index 8 g4 + l15 / 4 (+ 4), columns 4 (l15 % 4) .. + 3 of group e
#pragma unroll
  for (int e = 0; e < 4; ++e) col_at[e] = (8 * g4 + (l15 >> 2)) * 256 + 8 * (l15 & 3) + 32 * (e ^ (l15 >> 2));
  auto fragment = [&](bool col, const char* base, int side, int e) {
    if (col) {
      const char* p = base + col_at[e] + 128 * (side ^ (g4 & 1));
      const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p));
      const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p + 1024));
      typedef short s16x8_t __attribute__((ext_vector_type(8)));
      const s16x8_t both = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      return __builtin_bit_cast(bf16x8_t, both);
    }
    return *reinterpret_cast<const bf16x8_t*>(base + 4096 * side + row_at + 1024 * e);
  };

  f32x4_t acc[4][4];  // [n tile][m tile]
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // While step t is multiplied from registers, the operands of step t + 1 are read from LDS.  The barrier at the head of
  // step t: a wave's loads of step t + 1 are the oldest of those of steps t + 1 .. t + 4, four each, so after it everybody's
  // have landed; and everybody's reads of step t are complete (lgkmcnt), so the loads of step t + 5 may take its stage.
  bf16x8_t af[2][4], bf[2][4];
  auto read = [&](int set, int stage) {
    const char* sa = smem + stage * kPairStage;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      bf[set][e] = fragment(true, sa + kPairOperand, wn, e);
      af[set][e] = fragment(A_COL, sa, wm, e);
    }
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[set][j], af[set][i], acc[j][i], 0, 0, 0);
  };
#pragma unroll
  for (int p = 0; p < kPairStages; ++p) issue(t_begin + p, p);
  asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" ::: "memory");
  read(0, 0);
  int stage = 0;  // of step t
  auto step = [&](int t, int set) {
    asm volatile("s_waitcnt vmcnt(12) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    issue(t + kPairStages, stage);
    stage = stage == kPairStages - 1 ? 0 : stage + 1;
    read(set ^ 1, stage);
    multiply(set);
  };
  int t = t_begin;
  for (; t + 2 <= t_end; t += 2) {
    step(t, 0);
    step(t + 1, 1);
  }
  if (t < t_end) step(t, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // acc[j][i][v] = C[m0 + 64 wm + 16 i + l15][n0 + 64 wn + 16 j + 4 g4 + v]
  if constexpr (SPLIT) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + 64 * wm + 16 * i + l15;
      if (m >= g.M) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + 64 * wn + 16 * j + 4 * g4;
        if (n < g.N) *reinterpret_cast<f32x4_t*>(g.part + ((int64_t)blockIdx.y * g.M + m) * g.N + n) = acc[j][i];
      }
    }
  } else {
    __syncthreads();  // every wave has read its last step: the ring is free
    char* band = smem + wv * 8192;  // 64 rows x 128 bytes, chunk c of row r in slot c ^ (r & 7)
    const int nb = n0 + 64 * wn;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float b4[4] = {0.f, 0.f, 0.f, 0.f};
      if (g.bias && nb + 16 * j < g.N) {
        const u32x2_t b = *reinterpret_cast<const u32x2_t*>(g.bias + nb + 16 * j + 4 * g4);
        b4[0] = lo_of(b.x); b4[1] = hi_of(b.x); b4[2] = lo_of(b.y); b4[3] = hi_of(b.y);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * i + l15;
        u32x2_t o;
        o.x = pack_pair(acc[j][i][0] + b4[0], acc[j][i][1] + b4[1]);
        o.y = pack_pair(acc[j][i][2] + b4[2], acc[j][i][3] + b4[3]);
        *reinterpret_cast<u32x2_t*>(band + r * 128 + (((2 * j + (g4 >> 1)) ^ (r & 7)) << 4) + 8 * (g4 & 1)) = o;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int c = lane & 7;
    if (nb + 8 * c < g.N) {  // N % 8 == 0
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int r = 8 * t + (lane >> 3), m = m0 + 64 * wm + r;
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(band + r * 128 + ((c ^ (r & 7)) << 4));
        if (m < g.M) *reinterpret_cast<u32x4_t*>(g.C + (int64_t)m * g.N + nb + 8 * c) = v;
      }
    }
  }
#endif
}

// C = bf16(sum of the slices in order + bias), four columns per thread
__global__ __launch_bounds__(256) void gemm_mid_reduce_kernel(const float* __restrict__ part, int slices, int64_t quads, int nq,
                                                              const uint16_t* __restrict__ bias, uint16_t* __restrict__ C) {
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
  reinterpret_cast<u32x2_t*>(C)[e] = out;
}

struct MidPlan {
  int64_t tiles_m, tiles;
  int slices, steps;
  int rows;   // of a tile of gemm_mid_kernel (kind 2: 256, gemm_tn_kernel); 0: gemm_mid_pair_kernel
  int chain;  // steps of a chain, below `steps` where a whole contraction's chains are ended early
};
// gemm_mid_pair_kernel, and the most slices of either kernel (the workspace is sized before the kind is known): the split with
// the least of (steps of one workgroup) + (slabs written and read, one more launch), with the times measured on this kernel:
// 0.3 us a step when a CU has one workgroup (load latency), 0.22 us for each of two (LDS bandwidth), slabs at about 4 TB/s, 4 us
// for the reduction's launch.  Up to 128 tiles the slices stay within one workgroup per CU: past that the model says level and
// the extra slabs lose (this kernel at 1000 rows of 2048 x 8192, 128 tiles: 74 us whole, 52 in two slices, 60 in four; 200 x
// 4096 x 14336, 64 tiles: 46 in four, 51 in eight).
MidPlan plan_pair(int64_t M, int64_t N, int64_t K) {
  MidPlan p;
  p.rows = 0;
  p.tiles_m = (M + kPairTile - 1) / kPairTile;
  p.tiles = p.tiles_m * ((N + kPairTile - 1) / kPairTile);
  const int64_t nk = (K + 31) / 32;
  double best = 0;
  p.steps = (int)nk;
  p.slices = 1;
  for (int64_t s = 1; s <= 8 && s <= nk; ++s) {
    const int64_t steps = (nk + s - 1) / s, slices = (nk + steps - 1) / steps, per_cu = (p.tiles * slices + 255) / 256;
    if (slices > 1 && p.tiles <= 128 && p.tiles * slices > 256) break;
    const double t = (double)steps * (per_cu == 1 ? 0.3 : 0.22 * (double)per_cu) +
                     (slices > 1 ? 4.0 + 8e-6 / 4 * (double)slices * (double)M * (double)N : 0.0);
    if (s == 1 || t < best) {
      best = t;
      p.steps = (int)steps;
      p.slices = (int)slices;
    }
  }
  p.chain = p.steps;
  return p;
}

// No fp32 chain is longer than the split of plan_pair would make it, which one whole contraction in nine is (3696 products of
// kinds 0 and 1, 48 - 2047 rows): gemm_mid_kernel at 64 and 128 rows then ends its chains there, at 3 % of its time on average,
// and the others are no candidates (1183 x 3584 x 9728, from 256 rows to 128: 126 -> 140 us).
// Kinds 0 and 1: the kernel, tile height and split with the least modelled time in us, a term for each round of 256 workgroups
// (512 of the kernels that run two per CU), for its steps and for how full the chip is (its clock falls with the load), and for
// the slabs.  The terms are fitted to 760 products (40 - 8192 rows, the widths of seven model shapes), every tile and split of
// each measured; on 380 others the pick is 0.7 % slower than the fastest on average.
// Kind 2: gemm_mid_pair_kernel, or the 256 x 256 tiles of gemm_tn.hip, by the same kind of model (fitted to 260 products, 0.1 %
// slower than the faster one on average).  The wide tiles win from about half a round of them on (1000 tokens of 8192 x 2048
// 51.5 -> 31.3 us, 4096 x 4096 44.4 -> 30.6, of 2048 x 2048 15.1 and 21.9).  Where the model has them less than 5 % ahead they are
// up to 12 % behind (585 tokens of 4096 x 2048, 887 of 2560 x 3072 20.2 and 21.8) and seldom ahead (517 of 8192 x 1024, 18 %).
MidPlan plan_mid(int kind, int64_t M, int64_t N, int64_t K) {
  const MidPlan pair = plan_pair(M, N, K);
  MidPlan p = pair;
  if (kind == 2) {
    // whole contractions only: a slice's sums are shorter chains, and with few tiles the 256 x 256 ones are fewer still
    const double k = (double)((K + 31) / 32), tiles = (double)(((M + 255) / 256) * ((N + 255) / 256)), whole = ceil(tiles / 256),
                 rounds = (double)((pair.tiles + 255) / 256);
    const double wide = 0.2 + 7.26 * whole + k * (0.44 * whole + 0.25 * tiles / 256);
    const double narrow = 3.8 + 1.6 * rounds + k * (rounds > 1 ? 0.04 * rounds : 0.095) + 0.265 * k * (double)pair.tiles / 256;
    if (pair.slices == 1 && wide < 0.95 * narrow) p.rows = 256;
    return p;
  }
  double best = 1e30;
  if (kind == 1 && pair.slices == 1) {
    const double k = (double)((K + 31) / 32), rounds = (double)((pair.tiles + 255) / 256);
    best = 1.54 + 2.19 * rounds + k * (rounds > 1 ? 0.15 * rounds : 0.19) + 0.07 * k * (double)pair.tiles / 256;
  }
  const int64_t nk = K / kMidStep;
  for (const int rows : {64, 128, 256}) {
    const int64_t tiles_m = (M + rows - 1) / rows, tiles = tiles_m * ((N + kMidCols - 1) / kMidCols);
    for (int64_t s = 1; s <= (rows == 256 ? 1 : pair.slices) && s <= nk; ++s) {
      const int64_t steps = (nk + s - 1) / s, slices = (nk + steps - 1) / steps, items = tiles * slices;
      const double k = (double)steps, rounds = (double)((items + 255) / 256), pairs = (double)((items + 511) / 512),
                   fill = (double)items / 256, slabs = 1e-6 * (double)slices * (double)M * (double)N;
      double t = rows == 64    ? pairs * 3.74 + k * (rounds > 1 ? 0.53 * pairs : 0.35)
                 : rows == 128 ? rounds * (5.04 + 0.32 * k) + 0.14 * k * fill
                               : rounds * (8.72 + 0.32 * k) + 0.26 * k * fill;
      if (slices > 1) t += rows == 64 ? 2.23 + 2.71 * slabs : 3.84 + 1.84 * slabs;
      const bool fold = steps > pair.steps;
      if (t < best && !(fold && (rows == 256 || slices > 1))) {
        best = t;
        p.rows = rows;
        p.tiles_m = tiles_m;
        p.tiles = tiles;
        p.steps = (int)steps;
        p.slices = (int)slices;
        p.chain = !fold ? (int)steps : pair.steps > 3 ? pair.steps / 2 * 2 : 2;
      }
    }
  }
  return p;
}

// the wide tiles of kind 2 add no bias
MidPlan plan_of(int kind, bool bias, int64_t M, int64_t N, int64_t K) { return kind == 2 && bias ? plan_pair(M, N, K) : plan_mid(kind, M, N, K); }

// the LDS limit is a per-device attribute of the function
int reserve_lds(const void* fn, int bytes, bool (&set)[64]) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (dev >= 0 && set[dev]) return 0;
  const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return fail(TTAMD_ELAUNCH, "gemm_mid: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
  if (dev >= 0) set[dev] = true;
  return 0;
}

template <bool B_COL, bool SPLIT, int MT, int WGS, bool FOLD = false>
int launch_mid(MidArgs& g, hipStream_t s) {
  static bool set[64] = {};
  using S = MidShape<MT, WGS>;
  if (int rc = reserve_lds(reinterpret_cast<const void*>(&gemm_mid_kernel<B_COL, SPLIT, MT, WGS, FOLD>), S::lds, set)) return rc;
  g.per_xcd = (g.tiles * g.slices + 7) / 8;
  gemm_mid_kernel<B_COL, SPLIT, MT, WGS, FOLD><<<dim3(8u * g.per_xcd), dim3(512), S::lds, s>>>(g);
  return check_launch("gemm_mid");
}

template <bool B_COL>
int launch_rows(MidArgs& g, int rows, hipStream_t s) {
  if (rows == 256) return launch_mid<B_COL, false, 8, 1>(g, s);
  if (g.slices == 1 && g.chain < g.steps_per_slice) return rows == 128 ? launch_mid<B_COL, false, 4, 1, true>(g, s) : launch_mid<B_COL, false, 2, 2, true>(g, s);
  if (rows == 128) return g.slices > 1 ? launch_mid<B_COL, true, 4, 1>(g, s) : launch_mid<B_COL, false, 4, 1>(g, s);
  return g.slices > 1 ? launch_mid<B_COL, true, 2, 2>(g, s) : launch_mid<B_COL, false, 2, 2>(g, s);
}

template <bool A_COL, bool SPLIT>
int launch_pair(MidArgs& g, hipStream_t s) {
  static bool set[64] = {};
  if (int rc = reserve_lds(reinterpret_cast<const void*>(&gemm_mid_pair_kernel<A_COL, SPLIT>), kPairLds, set)) return rc;
  g.per_xcd = (g.tiles + 7) / 8;
  gemm_mid_pair_kernel<A_COL, SPLIT><<<dim3(8u * g.per_xcd, (unsigned)g.slices), dim3(256), kPairLds, s>>>(g);
  return check_launch("gemm_mid");
}

}  // namespace
}  // namespace ttamd

using namespace ttamd;

extern "C" size_t ttamd_gemm_mid_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const MidPlan p = plan_pair(M, N, K);
  return p.slices > 1 ? (size_t)p.slices * M * N * sizeof(float) : 0;
}

extern "C" int ttamd_gemm_mid_plan(int kind, int bias, int64_t M, int64_t N, int64_t K, int* tile_rows, int* slices, int* chain) {
  TT_REQUIRE(kind >= 0 && kind <= 2 && M > 0 && N > 0 && K > 0 && tile_rows && slices && chain, "gemm_mid_plan: bad argument");
  const MidPlan p = plan_of(kind, bias != 0, M, N, K);
  *tile_rows = p.rows;
  *slices = p.slices;
  *chain = 32 * p.chain;
  return TTAMD_OK;
}

extern "C" int ttamd_gemm_mid_bf16(int kind, const void* a, const void* b, const void* bias, void* c, int64_t M, int64_t N, int64_t K,
                                   void* workspace, size_t workspace_bytes, void* stream) {
  TT_REQUIRE(kind >= 0 && kind <= 2, "gemm_mid: unknown kind %d", kind);
  TT_REQUIRE(a && b && c && aligned16(a) && aligned16(b) && aligned16(c) && (!bias || (reinterpret_cast<uintptr_t>(bias) & 7u) == 0),
             "gemm_mid: operands must be non-null and 16-byte aligned (bias: 8)");
  TT_REQUIRE(M > 0 && N > 0 && K > 0 && N % 64 == 0 && (kind == 2 ? M % 64 == 0 : K % 64 == 0),
             "gemm_mid: bad shape M=%lld N=%lld K=%lld", (long long)M, (long long)N, (long long)K);
  // per-lane byte offsets inside the kernels are 32-bit
  TT_REQUIRE(M * N < (int64_t(1) << 30) && M * K < (int64_t(1) << 30) && N * K < (int64_t(1) << 30), "gemm_mid: operands too large");
  const MidPlan p = plan_of(kind, bias != nullptr, M, N, K);
  const size_t need = p.slices > 1 ? (size_t)p.slices * M * N * sizeof(float) : 0;
  if (need) {
    if (!workspace || workspace_bytes < need)
      return fail(TTAMD_EWORKSPACE, "gemm_mid: workspace of %zu bytes, %zu needed", workspace_bytes, need);
    TT_REQUIRE(aligned16(workspace), "gemm_mid: the workspace must be 16-byte aligned");
  }
  MidArgs g = {reinterpret_cast<const uint16_t*>(a), reinterpret_cast<const uint16_t*>(b), reinterpret_cast<const uint16_t*>(bias),
               reinterpret_cast<uint16_t*>(c), reinterpret_cast<float*>(workspace), (int)M, (int)N, (int)K, (int)p.tiles_m, (int)p.tiles, 0, p.slices, p.steps, p.chain};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (kind == 2 && p.rows) return run_gemm_tn(a, b, c, K, M, N, s);
  const int rc = p.rows ? (kind == 0 ? launch_rows<false>(g, p.rows, s) : launch_rows<true>(g, p.rows, s))
                 : kind == 1 ? launch_pair<false, false>(g, s)  // whole
                 : p.slices > 1 ? launch_pair<true, true>(g, s) : launch_pair<true, false>(g, s);
  if (rc || p.slices == 1) return rc;
  const int64_t quads = M * N / 4;
  gemm_mid_reduce_kernel<<<dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s>>>(g.part, p.slices, quads, g.N / 4, g.bias, g.C);
  return check_launch("gemm_mid: reduction");
}
