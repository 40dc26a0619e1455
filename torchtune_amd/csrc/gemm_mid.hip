// Plain bf16 products of a few dozen to some thousand rows: the three matmuls of a fake-quantised linear below the sizes of the
// 256 x 256-tile kernels (torchtune/modules: F.linear(fq(x), fq(W)) and what autograd derives from it).
//
//   kind 0   C[M, N] = A[M, K] . B[N, K]^T (+ bias)     forward
//   kind 1   C[M, N] = A[M, K] . B[K, N]                grad-input
//   kind 2   C[M, N] = A[K, M]^T . B[K, N]              weight gradient (the contraction runs over the tokens)
//
// At these sizes a product is a few dozen to a few hundred tiles of 128 x 128: what bounds it is the latency of a tile's
// contraction and how many CUs have one, not the matrix pipes.  Four waves (64 x 64 outputs each) per tile, two workgroups
// per CU; both operands go HBM -> LDS by direct loads into a ring of five stages of 32 contraction indices (80 KB), four steps
// ahead, one barrier per step, and from LDS to registers one step ahead of the MFMAs.  An operand that lies along the
// contraction is read from LDS as 16-byte pieces, one that lies across it through the transposing read
// (ds_read_b64_tr_b16); the 16-byte chunks of a stage are permuted on the global-address side of the loads so that the
// lanes served together fall on disjoint banks.  The 64 x 64 wave tile needs 128 bytes of LDS reads per cycle at the full
// matrix rate, so the kernel tops out near 850 TFLOP/s (1000 x 8192 x 2048, second kind: 40 us).
// Against the vendor library (its kernel alone, behind a queue of other products; choosing it costs 31 us of host time):
// 1000 x 2048 x 2048 forward 22.0 and 16.8 us, grad-input 22.4 and 21.1, weight gradient 17.8 and 23.3; 1000 x 2048 x 8192
// forward 51 and 51.  A training pass of a 1B-shaped layer over 1000 tokens with its 21 products: 1380 -> 830 us.
// Launches of few tiles cut the contraction into slices (fp32 slabs, added in slice order by gemm_mid_reduce_kernel).
#include "common.h"
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

struct MidArgs {
  const uint16_t* A;
  const uint16_t* B;
  const uint16_t* bias;  // [N] or null
  uint16_t* C;
  float* part;           // SPLIT: [slices, M, N]
  int M, N, K;
  int tiles_m, tiles, per_xcd;
  int steps_per_slice;
};

constexpr int kMidTile = 128;
constexpr int kMidOperand = 8192;              // 128 x 32 bf16
constexpr int kMidStage = 2 * kMidOperand;
constexpr int kMidStages = 5;
constexpr int kMidLds = kMidStages * kMidStage;

__device__ __constant__ u32x4_t kMidZero = {0, 0, 0, 0};

template <bool A_COL, bool B_COL, bool SPLIT>
__global__ __launch_bounds__(256, 2) void gemm_mid_kernel(const MidArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // workgroup ids go round-robin to the 8 XCDs: each gets a run of neighbouring tiles, row tiles first
  const int tile = (int)(blockIdx.x & 7) * g.per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= g.per_xcd || tile >= g.tiles) return;
  const int m0 = (tile % g.tiles_m) * kMidTile, n0 = (tile / g.tiles_m) * kMidTile;
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
  const int lda = A_COL ? g.M : g.K, ldb = B_COL ? g.N : g.K;
  offsets(0, A_COL, m0, g.M, lda);
  offsets(1, B_COL, n0, g.N, ldb);
  const int64_t a_step = A_COL ? (int64_t)lda * 64 : 64, b_step = B_COL ? (int64_t)ldb * 64 : 64;
  const bool ragged = (g.K & 31) != 0;  // only across the contraction on both sides (checked on the host)
  auto issue = [&](int t, int stage) {
    const int tk = t < t_end ? t : t_end - 1;  // past the end: the last step again (the waits count a fixed number in flight)
    const char* ab = reinterpret_cast<const char*>(g.A) + (int64_t)tk * a_step;
    const char* bb = reinterpret_cast<const char*>(g.B) + (int64_t)tk * b_step;
    const uint32_t sa = lds0 + stage * kMidStage + wv * 2048;
    if (A_COL && B_COL && ragged && tk == nk_all - 1) {
      const char* z = reinterpret_cast<const char*>(&kMidZero);
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const bool in = 32 * tk + krow[d] < g.K;
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(in ? ab + voff[0][d] : z), "s"(sa + 1024u * d) : "memory", "m0");
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(in ? bb + voff[1][d] : z), "s"(sa + kMidOperand + 1024u * d) : "memory", "m0");
      }
      return;
    }
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff[0][d]), "s"(ab), "s"(sa + 1024u * d) : "memory", "m0");
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff[1][d]), "s"(bb), "s"(sa + kMidOperand + 1024u * d) : "memory", "m0");
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
    const char* sa = smem + stage * kMidStage;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      bf[set][e] = fragment(B_COL, sa + kMidOperand, wn, e);
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
  for (int p = 0; p < kMidStages; ++p) issue(t_begin + p, p);
  asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" ::: "memory");
  read(0, 0);
  int stage = 0;  // of step t
  auto step = [&](int t, int set) {
    asm volatile("s_waitcnt vmcnt(12) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    issue(t + kMidStages, stage);
    stage = stage == kMidStages - 1 ? 0 : stage + 1;
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
};
// Slices of the contraction: the split with the least of (steps of one workgroup) + (slabs written and read, one more
// launch), with the times measured on this kernel: 0.3 us a step when a CU has one workgroup (load latency), 0.22 us for
// each of two (LDS bandwidth), slabs at about 4 TB/s, 4 us for the reduction's launch.  Up to 128 tiles the slices stay within
// one workgroup per CU: past that the model says level and the extra slabs lose (1000 rows of 2048 x 8192, 128 tiles: 74 us
// whole, 52 in two slices, 60 in four; 200 x 4096 x 14336, 64 tiles: 46 in four, 51 in eight).  Over 222 products of 53 - 8192
// rows and 256 - 14336 columns the split picked is 0.7 % slower than the fastest of 1 - 8 on average.
MidPlan plan_mid(int64_t M, int64_t N, int64_t K) {
  MidPlan p;
  p.tiles_m = (M + kMidTile - 1) / kMidTile;
  p.tiles = p.tiles_m * ((N + kMidTile - 1) / kMidTile);
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
  return p;
}

template <bool A_COL, bool B_COL>
int launch_mid(MidArgs& g, const MidPlan& p, hipStream_t s) {
  static bool attr_set[64] = {};  // the LDS limit is a per-device attribute of the function
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (dev < 0 || !attr_set[dev]) {
    for (const void* fn : {reinterpret_cast<const void*>(&gemm_mid_kernel<A_COL, B_COL, false>), reinterpret_cast<const void*>(&gemm_mid_kernel<A_COL, B_COL, true>)}) {
      const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kMidLds);
      if (e != hipSuccess) return fail(TTAMD_ELAUNCH, "gemm_mid: cannot reserve %d bytes of LDS: %s", kMidLds, hipGetErrorString(e));
    }
    if (dev >= 0) attr_set[dev] = true;
  }
  const dim3 grid((unsigned)(8 * g.per_xcd), (unsigned)p.slices), block(256);
  if (p.slices == 1) {
    gemm_mid_kernel<A_COL, B_COL, false><<<grid, block, kMidLds, s>>>(g);
    return check_launch("gemm_mid");
  }
  gemm_mid_kernel<A_COL, B_COL, true><<<grid, block, kMidLds, s>>>(g);
  if (int rc = check_launch("gemm_mid")) return rc;
  const int64_t quads = (int64_t)g.M * g.N / 4;
  gemm_mid_reduce_kernel<<<dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s>>>(g.part, p.slices, quads, g.N / 4, g.bias, g.C);
  return check_launch("gemm_mid: reduction");
}

}  // namespace
}  // namespace ttamd

using namespace ttamd;

extern "C" size_t ttamd_gemm_mid_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const MidPlan p = plan_mid(M, N, K);
  return p.slices > 1 ? (size_t)p.slices * M * N * sizeof(float) : 0;
}

extern "C" int ttamd_gemm_mid_bf16(int kind, const void* a, const void* b, const void* bias, void* c, int64_t M, int64_t N, int64_t K,
                                   void* workspace, size_t workspace_bytes, void* stream) {
  TT_REQUIRE(kind >= 0 && kind <= 2, "gemm_mid: unknown kind %d", kind);
  TT_REQUIRE(a && b && c && aligned16(a) && aligned16(b) && aligned16(c) && (!bias || (reinterpret_cast<uintptr_t>(bias) & 7u) == 0),
             "gemm_mid: operands must be non-null and 16-byte aligned (bias: 8)");
  TT_REQUIRE(M > 0 && N > 0 && K > 0 && N % 64 == 0 && (kind == 2 ? M % 64 == 0 : K % 64 == 0),
             "gemm_mid: bad shape M=%lld N=%lld K=%lld", (long long)M, (long long)N, (long long)K);
  // per-lane byte offsets inside the kernel are 32-bit
  TT_REQUIRE(M * N < (int64_t(1) << 30) && M * K < (int64_t(1) << 30) && N * K < (int64_t(1) << 30), "gemm_mid: operands too large");
  const MidPlan p = plan_mid(M, N, K);
  MidArgs g = {reinterpret_cast<const uint16_t*>(a), reinterpret_cast<const uint16_t*>(b), reinterpret_cast<const uint16_t*>(bias),
               reinterpret_cast<uint16_t*>(c), nullptr, (int)M, (int)N, (int)K, (int)p.tiles_m, (int)p.tiles, (int)((p.tiles + 7) / 8), p.steps};
  if (p.slices > 1) {
    const size_t need = ttamd_gemm_mid_workspace_bytes(M, N, K);
    if (!workspace || workspace_bytes < need)
      return fail(TTAMD_EWORKSPACE, "gemm_mid: workspace of %zu bytes, %zu needed", workspace_bytes, need);
    TT_REQUIRE(aligned16(workspace), "gemm_mid: the workspace must be 16-byte aligned");
    g.part = reinterpret_cast<float*>(workspace);
  }
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return kind == 0 ? launch_mid<false, false>(g, p, s) : kind == 1 ? launch_mid<false, true>(g, p, s) : launch_mid<true, true>(g, p, s);
}
