// Fused NF4-dequantise + bf16 MFMA GEMM, second generation: the weight operand never goes through LDS as bf16.
//
//     C[M, Nout] = X[M, Kc] . D(Wv)[Nout, Kc]^T  (+ bias)  + (lscale . lX)[M, R] . lW[Nout, R]^T
//
// `Wv` is a "weight view" whose rows are output columns and whose packed 4-bit codes run along the
// contraction dimension:
//   forward  : Wv = W   [N, K]  (the NF4 tensor as stored),   one scaler per row per 64 contraction elements
//   backward : Wv = W^T [K, N]  (a transposed copy of the codes), one scaler per contraction element per
//              64 output columns (NF4 blocks run along K, i.e. along the output columns of this view)
//
// This file: tiles of 256 x 256 for products of many rows, and the rules that send a product there, to the tiles of
// nf4_gemm_mid.hip or to the weight expanded once (nf4_gemm_dense.hip).
//
// Work split.  4 waves; wave w owns the 64 output columns [64w, 64w+64) of the tile for all its rows.  A lane of the MFMA weight
// operand needs 8 consecutive contraction elements of one output column: exactly one dword of codes.  Each lane expands its
// own code dwords in registers (byte -> pair of fp32 code points from a 256-entry LDS table, multiply by the scaler in fp32, round
// to bf16: bit-identical to the stand-alone dequantise kernel) one phase ahead of the MFMA that consumes them.
//
// Every global read of the main loop is a direct-to-LDS load (global_load_lds_*): the activation tile with an
// XOR swizzle applied on the global-address side, the code bytes and the scalers into wave-private slots.
// That keeps the vector-memory counter free of register-destination loads, so a single explicit
// `s_waitcnt vmcnt(one batch)` per k-step lets the next batch stay in flight (prefetch distance two k-steps;
// four activation stages so that one workgroup barrier per k-step suffices).
//
// This part is power-limited under matrix load and v_mfma_f32_16x16x32_bf16 sustains 13 % more FLOP/s than 32 x 32 x 16 at the same
// power (2.04 against 1.80 PFLOP/s for MFMA-only loops): a lane (l15, lg) of the weight operand holds row l15 of a 16-column
// tile and the 8 contraction elements [16 lg + 8 ks, + 8) of substep ks, and a 64-wide k-step is two substeps of NT (4) x MT (16)
// MFMAs.  The code bytes a direct-to-LDS instruction leaves as 16 bytes per (row, half) are read back as 8 bytes per (row,
// quarter), the activation operand is chunk 2 lg + ks of its row.
//   phase p = (substep ks = p / 2, half ih = p % 2): the NT x MT/2 MFMAs of substep ks against activation tiles
//     [MT/2 ih, + MT/2), the operand reads of the next phase, the finish of the 8 table entries fetched in the previous
//     phase and the fetch of the next 8 (tiles 0, 1 of a substep in one phase, tiles 2, 3 in the next);
//   the workgroup barrier of a k-step stands after phase 0: from phase 1 on the entries fetched belong to the next
//     k-step's codes, which are read back right after it.

#include "common.h"
#include "group.h"
#include "nf4_gemm_args.h"
#include "nf4_math.h"

namespace ttamd {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

__device__ __constant__ float kNF4Rs[16] = TT_NF4_TABLE;

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  bf16x2_t v;
  v.x = (__bf16)lo;
  v.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, v);
}

#define TT_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

constexpr int kBM = 256, kBN = 256;

// LDS: a ring of activation tiles (shared by the waves), a ring of 3 wave-private {code bytes, scalers} slots; the table is a
// static LDS object of 256 byte values x (fp32 nf4[hi nibble], fp32 nf4[lo nibble])
struct RsLayout {
  static constexpr int kStageA = kBM * 128;  // activation tile: rows x 64 bf16
  static constexpr int kAStages = 4;
  static constexpr int kWOff = kAStages * kStageA;
  static constexpr int kStageW = 8192 + 2048;  // code bytes [wave][tile j][lane] x 16 B, then scalers [wave] x 512 B
  static constexpr int kWStages = 3;
  static constexpr int kTotal = kWOff + kWStages * kStageW;
};

// MODE 0: one scaler per (output column, 64-wide k-step), scaler tensor laid out like the weight's blocks
// MODE 2: the same scalers, tensor transposed so that the 64 columns of a wave are contiguous (one coalesced load)
// MODE 1: one scaler per contraction element, shared by the wave's 64 columns (the transposed weight of the backward)
template <int MODE>
__global__ __launch_bounds__(256) void nf4_gemm_rs16_kernel(const RsArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr bool PER_ELEM = MODE == 1;
  constexpr bool SCAL_T = MODE == 2;
  using L = RsLayout;
  constexpr int BM = kBM;
  constexpr int MT = BM / 16;       // 16-row activation tiles (MFMA columns) per wave
  constexpr int MH = MT / 2;        // of which a phase takes half
  constexpr int NT = 4;             // 16-column weight tiles (MFMA rows) per wave
  constexpr int ND = 2;             // direct-to-LDS instructions per k-step for the wave's code bytes (32 rows each)
  constexpr int kALoads = BM / 32;  // and for its share of the activation tile (8 rows each)
  constexpr int kBatch = kALoads + ND + (MODE == 0 ? ND : 1);
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, h = lane >> 5;    // roles on the load side
  const int l15 = lane & 15, lg = lane >> 4;   // roles on the MFMA side

  int tile_m, tile_n;
  {
    // workgroup ids are dealt round-robin to the 8 XCDs (one L2 each): give every XCD a band of m-tiles and walk it
    // column by column, so the workgroups resident on an XCD share each weight tile through its L2
    const int id = blockIdx.x;
    if ((g.tiles_m & 7) == 0) {
      const int xcd = id & 7, slot = id >> 3, band = g.tiles_m >> 3;
      tile_m = xcd * band + slot % band;
      tile_n = slot / band;
    } else {
      tile_m = id / g.tiles_n;
      tile_n = id % g.tiles_n;
    }
  }
  const int m0 = tile_m * BM, n0 = tile_n * kBN;
  const int Kc = g.Kc, nk = Kc >> 6;

  __shared__ float2 lut_s[256];
  lut_s[tid] = make_float2(round_to_bf16(kNF4Rs[tid >> 4]), round_to_bf16(kNF4Rs[tid & 15]));
  const char* lut = reinterpret_cast<const char*>(lut_s);

  // ---- activation tile.  A row is eight 16-byte chunks; chunk c of row r is stored in slot c ^ ((r >> 1) & 7), which
  //      makes the 128-bit operand reads below bank-conflict free.  A direct-to-LDS instruction writes lane l to
  //      linear slot l, so the lane fetches the chunk that belongs there.
  //      Weight view rows of this lane: piece j -> output column n0 + 64 wv + 32 j + l31; half h owns code bytes [16h, 16h+16).
  const int a_r8 = lane >> 3;
  uint32_t a_off[kALoads];
  uint32_t w_off[ND], s_off[ND];
#pragma unroll
  for (int i = 0; i < kALoads; ++i) {
    const int trow = wv * (BM / 4) + 8 * i + a_r8;
    const int chunk = (lane & 7) ^ ((trow >> 1) & 7);
    int row = m0 + trow;
    row = row < g.M ? row : g.M - 1;
    a_off[i] = ((uint32_t)row * (uint32_t)Kc + chunk * 8) * 2u;
  }
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    int col = n0 + wv * 64 + 32 * j + l31;
    col = col < g.Nout ? col : g.Nout - 1;
    w_off[j] = (uint32_t)(((int64_t)col * Kc) >> 1) + 16 * h;
    s_off[j] = (uint32_t)col * (uint32_t)(Kc >> 6) * 4u;
  }
  if constexpr (SCAL_T) {
    int col = n0 + wv * 64 + lane;
    col = col < g.Nout ? col : g.Nout - 1;
    s_off[0] = (uint32_t)col * 4u;
  }
  if constexpr (PER_ELEM) {
    int ob = (n0 >> 6) + wv;
    const int nob = g.Nout >> 6;
    ob = ob < nob ? ob : nob - 1;
    s_off[0] = ((uint32_t)ob * (uint32_t)Kc + lane) * 4u;
  }

  auto dma16 = [&](uint32_t voff, const char* base, uint32_t lds, int imm) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 ::"v"(voff), "s"(base), "s"(lds), "n"(imm) : "memory", "m0", "scc");
  };
  auto dma4 = [&](uint32_t voff, const char* base, uint32_t lds, int imm) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 ::"v"(voff), "s"(base), "s"(lds), "n"(imm) : "memory", "m0", "scc");
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)TT_LDS_PTR(smem);
  struct BatchAddr {
    const char *xb, *cb, *sb;
    uint32_t abase, wcodes, wscal;
  };
  const int64_t s_stride = PER_ELEM ? 256 : SCAL_T ? (int64_t)g.Nout * 4 : 4;
  auto batch_addr_at = [&](const char* xb, const char* cb, const char* sb, int sa, int sw) -> BatchAddr {
    BatchAddr b;
    b.xb = xb;
    b.cb = cb;
    b.sb = sb;
    b.abase = lds0 + sa * L::kStageA + wv * (BM / 4) * 128;
    b.wcodes = lds0 + L::kWOff + sw * L::kStageW + wv * ND * 1024;
    b.wscal = lds0 + L::kWOff + sw * L::kStageW + 8192 + wv * 512;
    return b;
  };
  auto batch_addr = [&](int t, int sa, int sw) -> BatchAddr {
    const int tk = t < nk ? t : nk - 1;
    return batch_addr_at(reinterpret_cast<const char*>(g.X) + ((int64_t)tk << 7),
                         reinterpret_cast<const char*>(g.codes) + ((int64_t)tk << 5),
                         reinterpret_cast<const char*>(g.scal) + tk * s_stride, sa, sw);
  };
  auto issue_one = [&](const BatchAddr& b, int d) {
    if (d < kALoads) {
      dma16(a_off[d], b.xb, b.abase, d * 1024);
    } else if (d < kALoads + ND) {
      const int j = d - kALoads;
      dma16(w_off[j], b.cb, b.wcodes, j * 1024);
    } else if (d < kBatch) {
      const int j = d - kALoads - ND;
      dma4(s_off[j], b.sb, b.wscal, j * 256);
    }
  };
  auto issue = [&](int t, int sa, int sw) {
    const BatchAddr b = batch_addr(t, sa, sw);
#pragma unroll
    for (int d = 0; d < kBatch; ++d) issue_one(b, d);
  };

  // ---- weights: tile j is rows 16 j + l15 of the wave's 64; substep ks of this lane is code dword 2 lg + ks of the
  //      row's eight.  A load instruction left row 32 J + r, bytes [16 H, + 16) at lane r + 32 H of piece J.
  uint32_t codes[NT][2];
  float sc[NT], sc_next[NT];
  float2 pend[2][4];  // the eight table entries in flight: [tile of the pair][code byte]
  u32x4_t wfa[NT], wfb[NT];
  bf16x8_t xfa[MH], xfb[MH];

  auto fetch_byte = [&](int jj, int j, int ks, int b) {
    uint32_t off;
    if (b == 0) {
      asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_0"
          : "=v"(off) : "v"(3u), "v"(codes[j][ks]));
    } else {
      off = ((codes[j][ks] >> (8 * b)) & 0xffu) << 3;
    }
    pend[jj][b] = *reinterpret_cast<const float2*>(lut + off);
  };
  auto finish_byte = [&](u32x4_t (&wf)[NT], int jj, int j, int b, const float (&s)[NT], const float (&s8)[8]) {
    if constexpr (PER_ELEM)
      wf[j][b] = pack_bf16x2(pend[jj][b].x * s8[2 * b], pend[jj][b].y * s8[2 * b + 1]);
    else
      wf[j][b] = pack_bf16x2(pend[jj][b].x * s[j], pend[jj][b].y * s[j]);
  };
  auto load_s8 = [&](float (&s8)[8], int sw, int ks) {
    if constexpr (PER_ELEM) {
      const f32x4_t* sp = reinterpret_cast<const f32x4_t*>(smem + L::kWOff + sw * L::kStageW + 8192 + wv * 512 + (16 * lg + 8 * ks) * 4);
      const f32x4_t a = sp[0], b = sp[1];
      s8[0] = a.x; s8[1] = a.y; s8[2] = a.z; s8[3] = a.w; s8[4] = b.x; s8[5] = b.y; s8[6] = b.z; s8[7] = b.w;
    }
  };
  auto load_codes = [&](int sw, float (&s_out)[NT]) {
    const char* wbase = smem + L::kWOff + sw * L::kStageW;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const u32x2_t v = *reinterpret_cast<const u32x2_t*>(wbase + (wv * ND + (j >> 1)) * 1024 +
                                                          (16 * (j & 1) + l15 + 32 * (lg >> 1)) * 16 + 8 * (lg & 1));
      codes[j][0] = v.x; codes[j][1] = v.y;
      if constexpr (MODE == 0) s_out[j] = *reinterpret_cast<const float*>(wbase + 8192 + wv * 512 + (j >> 1) * 256 + (16 * (j & 1) + l15) * 4);
      if constexpr (SCAL_T) s_out[j] = *reinterpret_cast<const float*>(wbase + 8192 + wv * 512 + (16 * j + l15) * 4);
    }
  };

  f32x4_t acc[NT][MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[j][i][v] = 0.f;

  // operand read offsets inside a stage: row 16 i + l15, chunk 2 lg + ks, slot = chunk ^ ((row >> 1) & 7)
  int x_off[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) x_off[ks] = l15 * 128 + (((2 * lg + ks) ^ ((l15 >> 1) & 7)) << 4);

  // One phase, in quarters.  Quarter q:
  //   MFMAs of weight tile q against the MH activation tiles of the phase's half
  //   operand reads of the NEXT phase: activation tiles [MH/4 q, + MH/4) of its half
  //   finish + fetch of code bytes 2 (q % 2), 2 (q % 2) + 1 of tile q / 2 of the pair (finish: what the previous phase
  //     fetched, into wf_next of the pair jp_fin; fetch: the pair jp_fetch of substep ks_fetch)
  //   up to two direct-to-LDS loads of batch `b`
  auto phase = [&](const bf16x8_t (&xf_use)[MH], int ih_use, const u32x4_t (&wf_use)[NT], bf16x8_t (&xf_next)[MH], int st_next,
                   int ks_next, int ih_next, u32x4_t (&wf_next)[NT], int jp_fin, const float (&s_fin)[NT], int sw_fin, int ks_fin,
                   int jp_fetch, int ks_fetch, const BatchAddr& b, int d_first, int d_even, int d_odd) {
    float s8[8];
    load_s8(s8, sw_fin, ks_fin);
    const char* sA = smem + st_next * L::kStageA + (MH * ih_next) * 2048;
    int d = d_first;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int nd = (q & 1) ? d_odd : d_even;
      const int jj = q >> 1, b0 = 2 * (q & 1);
      // The MFMAs are written in assembly with the accumulator tied to itself in the AGPR file: left to the register
      // allocator, the 64 four-register accumulators of this loop get different source and destination registers and are
      // copied around the loop's back edge (700 v_accvgpr moves per k-step).  The scheduler does not know such a
      // statement for a matrix instruction, so the interleaving is spelled out: one MFMA, one piece of the quarter's
      // other work, a scheduling barrier.  A 16 x 16 x 32 MFMA keeps the pipe for 16 cycles and the wave issues in
      // order: whatever follows it in program order rides in the 12 cycles before the next one can start.
      auto mfma = [&](int i) {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[q][MH * ih_use + i]) : "v"(wf_use[q]), "v"(xf_use[i]));
      };
      auto other = [&](int slot) {  // the quarter's other work in eight pieces
        constexpr int kReads = MH / 4;  // operand reads of the next phase per quarter: 2 (BM = 256) or 1
        switch (slot) {
          case 0:
            xf_next[kReads * q] = *reinterpret_cast<const bf16x8_t*>(sA + (kReads * q) * 2048 + x_off[ks_next]);
            break;
          case 1: finish_byte(wf_next, jj, 2 * jp_fin + jj, b0, s_fin, s8); break;
          case 2: fetch_byte(jj, 2 * jp_fetch + jj, ks_fetch, b0); break;
          case 3:
            if (kReads > 1) xf_next[kReads * q + 1] = *reinterpret_cast<const bf16x8_t*>(sA + (kReads * q + 1) * 2048 + x_off[ks_next]);
            break;
          case 4: finish_byte(wf_next, jj, 2 * jp_fin + jj, b0 + 1, s_fin, s8); break;
          case 5: fetch_byte(jj, 2 * jp_fetch + jj, ks_fetch, b0 + 1); break;
          case 6:
            if (nd > 0) issue_one(b, d);
            break;
          default:
            if (nd > 1) issue_one(b, d + 1);
            break;
        }
      };
      constexpr int kPer = 8 / MH;  // pieces per MFMA: 1 (BM = 256) or 2
#pragma unroll
      for (int i = 0; i < MH; ++i) {
        mfma(i);
#pragma unroll
        for (int u = 0; u < kPer; ++u) other(kPer * i + u);
        __builtin_amdgcn_sched_barrier(0);
      }
      d += nd;
    }
  };

  // ---- software pipeline: activation tile t in A stage t % 4, this wave's codes in W stage
  //      t % 3 (batch t + 2 issued during phases 0 and 1 of step t), with the barrier of step t after phase 0.  There
  //      this wave's batch t + 1 has landed (it was issued a step ago; the loads phase 0 just issued may be in flight)
  //      and, past the barrier, everybody's.  A wave that issues batch t + 2 into the A stage of tile t - 2 has passed
  //      barrier t - 1, which every wave reaches only after its last read of tile t - 2.
  const char *pxb, *pcb, *psb;
  issue(0, 0, 0);
  issue(1, 1, 1);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kBatch) : "memory");  // batch 0 landed everywhere, table written
  load_codes(0, sc);
  {
    // substep 0 in full, and the first pair of substep 1 on its way
    float s8[8];
    load_s8(s8, 0, 0);
#pragma unroll
    for (int jp = 0; jp < 2; ++jp) {
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int b = 0; b < 4; ++b) fetch_byte(jj, 2 * jp + jj, 0, b);
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int b = 0; b < 4; ++b) finish_byte(wfa, jj, 2 * jp + jj, b, sc, s8);
    }
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
#pragma unroll
      for (int b = 0; b < 4; ++b) fetch_byte(jj, jj, 1, b);
  }
#pragma unroll
  for (int i = 0; i < MH; ++i) xfa[i] = *reinterpret_cast<const bf16x8_t*>(smem + i * 2048 + x_off[0]);

  constexpr int kDEven = (kBatch + 7) / 8 > 1 ? 2 : 1;
  constexpr int kDOdd = (kBatch - 4 * kDEven + 3) / 4;
  static_assert(4 * kDEven + 4 * kDOdd >= kBatch && kDOdd <= 2 && kDOdd >= 0, "batch does not fit the 8 quarter phases");
  constexpr int kInPhase0 = 2 * (kDEven + kDOdd) < kBatch ? 2 * (kDEven + kDOdd) : kBatch;  // loads phase 0 issues
  int a0 = 0, w0 = 0;
  auto k_step = [&](int64_t adv) {
    const int a1 = (a0 + 1) & 3, a2 = (a0 + 2) & 3;
    const int w1 = w0 == 2 ? 0 : w0 + 1, w2 = w1 == 2 ? 0 : w1 + 1;
    const BatchAddr b = batch_addr_at(pxb, pcb, psb, a2, w2);
    pxb += adv << 7;
    pcb += adv << 5;
    psb += adv * s_stride;
    //    use        use   next operands          builds  finish: pair, scalers, stage, substep   fetch: pair, substep
    phase(xfa, 0, wfa, xfb, a0, 0, 1, wfb, 0, sc, w0, 1, 1, 1, b, 0, kDEven, kDOdd);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kInPhase0) : "memory");
    load_codes(w1, sc_next);
    phase(xfb, 1, wfa, xfa, a0, 1, 0, wfb, 1, sc, w0, 1, 0, 0, b, kInPhase0, kDEven, kDOdd);
    phase(xfa, 0, wfb, xfb, a0, 1, 1, wfa, 0, sc_next, w1, 0, 1, 0, b, kBatch, 0, 0);
    phase(xfb, 1, wfb, xfa, a1, 0, 0, wfa, 1, sc_next, w1, 0, 0, 1, b, kBatch, 0, 0);
#pragma unroll
    for (int j = 0; j < NT; ++j) sc[j] = sc_next[j];
    a0 = a1;
    w0 = w1;
  };
  const BatchAddr b2 = batch_addr(2, 0, 0);  // global bases of the next batch, carried through the loop
  pxb = b2.xb; pcb = b2.cb; psb = b2.sb;
  for (int kt = 0; kt < nk; ++kt) k_step(kt + 3 < nk ? 1 : 0);

  // the clamped batches issued by the last two steps; and the last MFMAs of the loop (assembly: the compiler does not
  // know they are matrix instructions) have left the pipeline before anything reads their accumulators
  asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
  // ---- adapter: one MFMA step per 32 ranks, operands straight from global memory; lane (l15, lg) holds ranks
  //      rc + 8 lg .. + 7 of weight column / activation row l15 of its tile
  if (g.lX != nullptr) {
    const uint16_t* __restrict__ lX = g.lX;
    const uint16_t* __restrict__ lW = g.lW;
    const int R = g.R;
    for (int rc = 0; rc < R; rc += 32) {
      const int r0 = rc + 8 * lg;
      const bool in = r0 < R;  // R % 8 == 0: a lane's 8 indices are all in or all out
      bf16x8_t wfr[NT];
      // the requests of half a step first, then their uses: two trips to memory per step (with the scaling between two
      // loads the compiler waited for each of them in turn)
      u32x4_t xraw[MH];
      auto load_x = [&](int ih) {
#pragma unroll
        for (int i = 0; i < MH; ++i) {
          int row = m0 + 16 * (MH * ih + i) + l15;
          row = row < g.M ? row : g.M - 1;
          xraw[i] = u32x4_t{0, 0, 0, 0};
          if (in) xraw[i] = *reinterpret_cast<const u32x4_t*>(lX + (int64_t)row * g.ldlx + r0);
        }
      };
      load_x(0);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        int col = n0 + wv * 64 + 16 * j + l15;
        col = col < g.Nout ? col : g.Nout - 1;
        u32x4_t raw = {0, 0, 0, 0};
        if (in) {
          if (g.lw_row_major) {
            raw = *reinterpret_cast<const u32x4_t*>(lW + (int64_t)col * R + r0);
          } else {
            uint32_t e[8];
#pragma unroll
            for (int d = 0; d < 8; ++d) e[d] = lW[(int64_t)(r0 + d) * g.Nout + col];
#pragma unroll
            for (int d = 0; d < 4; ++d) raw[d] = e[2 * d] | (e[2 * d + 1] << 16);
          }
        }
        wfr[j] = __builtin_bit_cast(bf16x8_t, raw);
      }
#pragma unroll
      for (int ih = 0; ih < 2; ++ih) {
        bf16x8_t xfr[MH];
        if (ih == 1) load_x(1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < MH; ++i) {
          u32x4_t raw = xraw[i];
          if (g.lscale != 1.0f) {
#pragma unroll
            for (int d = 0; d < 4; ++d)
              raw[d] = pack_bf16x2(bits_f32(raw[d] << 16) * g.lscale, bits_f32(raw[d] & 0xffff0000u) * g.lscale);
          }
          xfr[i] = __builtin_bit_cast(bf16x8_t, raw);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int i = 0; i < MH; ++i)
            acc[j][MH * ih + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wfr[j], xfr[i], acc[j][MH * ih + i], 0, 0, 0);
      }
    }
  }

  // ---- epilogue.  acc[j][i][v] = C[m][n] with m = m0 + 16 i + l15 and n = n0 + 64 wv + 16 j + 4 lg + v.
  __syncthreads();                      // every wave is done reading the activation ring
  if (n0 + wv * 64 >= g.Nout) return;  // the whole 64-column band of this wave lies outside (no barrier follows)
  {
    // each wave transposes its BM x 64 band through LDS (BM x 128 bytes per wave) and writes whole 128-byte row
    // segments; 16-byte chunk c of row r sits in slot c ^ (r & 7)
    char* band = smem + wv * (BM * 128);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      float b4[4] = {0.f, 0.f, 0.f, 0.f};
      if (g.bias) {
        const u32x2_t bb = *reinterpret_cast<const u32x2_t*>(g.bias + n0 + wv * 64 + 16 * j + 4 * lg);
        b4[0] = bits_f32(bb.x << 16); b4[1] = bits_f32(bb.x & 0xffff0000u);
        b4[2] = bits_f32(bb.y << 16); b4[3] = bits_f32(bb.y & 0xffff0000u);
      }
      float c4[4] = {1.f, 1.f, 1.f, 1.f};
      if (g.cscale) {
        const u32x2_t cc = *reinterpret_cast<const u32x2_t*>(g.cscale + n0 + wv * 64 + 16 * j + 4 * lg);
        c4[0] = bits_f32(cc.x << 16); c4[1] = bits_f32(cc.x & 0xffff0000u);
        c4[2] = bits_f32(cc.y << 16); c4[3] = bits_f32(cc.y & 0xffff0000u);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int r = 16 * i + l15;
        u32x2_t o;
        o.x = pack_bf16x2((acc[j][i][0] + b4[0]) * c4[0], (acc[j][i][1] + b4[1]) * c4[1]);
        o.y = pack_bf16x2((acc[j][i][2] + b4[2]) * c4[2], (acc[j][i][3] + b4[3]) * c4[3]);
        *reinterpret_cast<u32x2_t*>(band + r * 128 + (((2 * j + (lg >> 1)) ^ (r & 7)) << 4) + 8 * (lg & 1)) = o;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int c = lane & 7;
    uint16_t* crow = g.C + n0 + wv * 64 + 8 * c;
#pragma unroll 8
    for (int t = 0; t < BM / 8; ++t) {
      const int r = 8 * t + (lane >> 3);
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(band + r * 128 + ((c ^ (r & 7)) << 4));
      if (m0 + r < g.M) *reinterpret_cast<u32x4_t*>(crow + (int64_t)(m0 + r) * g.Nout) = v;
    }
  }
#endif
}

// The grouped grad-input on tiles of 256 x 256: the contraction runs through the members' segments (RsSegs).  With v_mfma_f32_32x32x16:
// a lane (l31, h) holds row l31 of a 32-column tile and the contraction elements [32 h + 8 ks, + 8) of substep ks (the 16 x 16 x 32 loop
// above spills with segments).  From a full round of these tiles on it is ahead of nf4_gemm_mid_kernel (14336 + 14336 rows of 4096
// at 8192 tokens, adapters and all: 1704 against 1940 us; at 4096 886 and 1004).
__global__ __launch_bounds__(256) void nf4_gemm_rs_segments_kernel(const RsArgs g, const RsSegs sg) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses LDS address-space casts and gfx950 builtins the host pass cannot parse
  using L = RsLayout;
  constexpr int BM = kBM;
  constexpr int MT = BM / 32;       // activation tiles (MFMA columns) per wave
  constexpr int NT = 2;             // weight tiles (MFMA rows) per wave
  constexpr int kALoads = BM / 32;  // direct-to-LDS instructions per wave per k-step for the activation tile (8 rows each)
  constexpr int kBatch = kALoads + NT + 1;  // vector-memory operations per wave per k-step
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, h = lane >> 5;

  int tile_m, tile_n;
  {
    const int id = blockIdx.x;
    if ((g.tiles_m & 7) == 0) {
      const int xcd = id & 7, slot = id >> 3, band = g.tiles_m >> 3;
      tile_m = xcd * band + slot % band;
      tile_n = slot / band;
    } else {
      tile_m = id / g.tiles_n;
      tile_n = id % g.tiles_n;
    }
  }
  const int m0 = tile_m * BM, n0 = tile_n * kBN;
  int nk = 0;  // k-steps of the whole contraction
  for (int q = 0; q < sg.n; ++q) nk += sg.Kc[q] >> 6;

  // ---- table: entry(byte) = (nf4[byte >> 4], nf4[byte & 15]) as two fp32 (each exactly a bf16 value)
  //      It is a separate LDS object so that the compiler can tell table reads from the direct-to-LDS destinations.
  __shared__ float2 lut_s[256];
  lut_s[tid] = make_float2(round_to_bf16(kNF4Rs[tid >> 4]), round_to_bf16(kNF4Rs[tid & 15]));
  const char* lut = reinterpret_cast<const char*>(lut_s);

  // ---- activation tile.  A row is eight 16-byte chunks; chunk c of row r is stored in slot c ^ ((r >> 1) & 7), which
  //      makes the 128-bit operand reads below bank-conflict free.  A direct-to-LDS instruction writes lane l to
  //      linear slot l, so the lane fetches the chunk that belongs there.
  const int a_r8 = lane >> 3;
  uint32_t a_off[kALoads];  // byte offset of this lane's chunk from X + k0
  // ---- weight view rows of this lane: tile j -> output column n0 + 64 wv + 32 j + l31; half h owns code bytes [16h, 16h+16)
  uint32_t w_off[NT], s_off;  // byte offsets from codes + k0/2 and from scal + tk
  // (the offsets depend on the row length kc of a segment's operands)
  auto set_offsets = [&](int kc) {
#pragma unroll
    for (int i = 0; i < kALoads; ++i) {
      const int trow = wv * (BM / 4) + 8 * i + a_r8;  // row inside the tile
      const int chunk = (lane & 7) ^ ((trow >> 1) & 7);
      int row = m0 + trow;
      row = row < g.M ? row : g.M - 1;
      a_off[i] = ((uint32_t)row * (uint32_t)kc + chunk * 8) * 2u;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      int col = n0 + wv * 64 + 32 * j + l31;
      col = col < g.Nout ? col : g.Nout - 1;
      w_off[j] = (uint32_t)(((int64_t)col * kc) >> 1) + 16 * h;
    }
    {
      // scalers of the wave's 64-column block for the 64 contraction elements of a k-step: lane l fetches element l
      int ob = (n0 >> 6) + wv;
      const int nob = g.Nout >> 6;
      ob = ob < nob ? ob : nob - 1;
      s_off = ((uint32_t)ob * (uint32_t)kc + lane) * 4u;
    }
  };
  set_offsets(sg.Kc[0]);

  // Direct-to-LDS loads are written as inline assembly: `voff` is this lane's 32-bit byte offset from the uniform
  // `base`, the wave's 64 lanes land in LDS at `lds`, `lds` + size, ...  Issued this way the compiler keeps no
  // bookkeeping for them (it would otherwise wait for ALL outstanding loads before the next LDS read it cannot prove
  // disjoint); completion is awaited explicitly with s_waitcnt vmcnt below.
  // M0 (the LDS destination) is formed by the scalar add itself: `lds` is a wave-uniform base, `imm` a compile-time
  // offset.  One wait state must separate a scalar write of M0 from the load that reads it.
  auto dma16 = [&](uint32_t voff, const char* base, uint32_t lds, int imm) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 ::"v"(voff), "s"(base), "s"(lds), "n"(imm) : "memory", "m0", "scc");
  };
  auto dma4 = [&](uint32_t voff, const char* base, uint32_t lds, int imm) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 ::"v"(voff), "s"(base), "s"(lds), "n"(imm) : "memory", "m0", "scc");
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)TT_LDS_PTR(smem);
  // A batch (k-step t) is kBatch loads: the activation tile -> A stage, this wave's code bytes and scalers -> W stage.
  // They are issued one at a time between MFMAs (slot d of the batch), never back to back: the address unit takes
  // tens of cycles per 64-lane load and a wave that finds its queue full cannot issue anything else meanwhile.
  struct BatchAddr {
    const char *xb, *cb, *sb;
    uint32_t abase, wcodes, wscal;  // LDS bases of this wave's share of the A stage, of its code bytes and of its scalers
  };
  // Global bases of k-step t are base + min(t, nk - 1) * stride (past the end the last tile is reloaded, never
  // consumed).  The main loop carries the three pointers and bumps them by a constant instead of recomputing them.
  auto batch_addr_at = [&](const char* xb, const char* cb, const char* sb, int sa, int sw) -> BatchAddr {
    BatchAddr b;
    b.xb = xb;
    b.cb = cb;
    b.sb = sb;
    b.abase = lds0 + sa * L::kStageA + wv * (BM / 4) * 128;
    b.wcodes = lds0 + L::kWOff + sw * L::kStageW + wv * NT * 1024;
    b.wscal = lds0 + L::kWOff + sw * L::kStageW + 8192 + wv * 512;
    return b;
  };
  auto issue_one = [&](const BatchAddr& b, int d) {  // d is a compile-time constant after unrolling
    if (d < kALoads) {
      dma16(a_off[d], b.xb, b.abase, d * 1024);
    } else if (d < kALoads + NT) {
      const int j = d - kALoads;
      dma16(w_off[j], b.cb, b.wcodes, j * 1024);
    } else if (d < kBatch) {
      dma4(s_off, b.sb, b.wscal, 0);
    }
  };
  // weights of one k-substep: a code byte -> one fp32 pair from the table (fetch), scaled and rounded to bf16 (finish)
  uint32_t codes[NT][4];  // this lane's code dwords of the k-step being expanded: [tile][k-substep]
  float2 pend[NT][4];     // table entries fetched in one phase, finished in the next: [tile][code byte]
  u32x4_t wfa[NT], wfb[NT];  // weight operands (8 bf16 each) of two consecutive k-substeps
  bf16x8_t xfa[MT], xfb[MT];

  auto fetch_byte = [&](int j, int ks, int b) {
    uint32_t off;
    if (b == 0) {
      // byte 0 as one sub-dword-addressed shift, like the compiler's own choice for bytes 1-3 (it would otherwise
      // emit a mask and a shift here)
      asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_0"
          : "=v"(off) : "v"(3u), "v"(codes[j][ks]));
    } else {
      off = ((codes[j][ks] >> (8 * b)) & 0xffu) << 3;
    }
    pend[j][b] = *reinterpret_cast<const float2*>(lut + off);
  };
  // finish byte b of tile j into wf[j]; s8 = the eight scalers of the substep
  auto finish_byte = [&](u32x4_t (&wf)[NT], int j, int b, const float (&s8)[8]) {
    wf[j][b] = pack_bf16x2(pend[j][b].x * s8[2 * b], pend[j][b].y * s8[2 * b + 1]);
  };
  auto load_s8 = [&](float (&s8)[8], int sw, int ks) {
    const f32x4_t* sp = reinterpret_cast<const f32x4_t*>(smem + L::kWOff + sw * L::kStageW + 8192 + wv * 512 + (32 * h + 8 * ks) * 4);
    const f32x4_t a = sp[0], b = sp[1];
    s8[0] = a.x; s8[1] = a.y; s8[2] = a.z; s8[3] = a.w; s8[4] = b.x; s8[5] = b.y; s8[6] = b.z; s8[7] = b.w;
  };
  auto load_codes = [&](int sw) {
    const char* wbase = smem + L::kWOff + sw * L::kStageW;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(wbase + (wv * NT + j) * 1024 + lane * 16);
      codes[j][0] = v.x; codes[j][1] = v.y; codes[j][2] = v.z; codes[j][3] = v.w;
    }
  };

  f32x16_t acc[NT][MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.f;

  // operand read offsets inside a stage: row 32 i + l31, chunk 4h + ks, slot = chunk ^ ((row >> 1) & 7)
  int x_off[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) x_off[ks] = l31 * 128 + (((4 * h + ks) ^ ((l31 >> 1) & 7)) << 4);

  // One phase = the 16 (NT x MT) MFMAs of a k-substep, cut into quarters.  Quarter q:
  //   MFMAs of weight tile q/2 against activation tiles [MT/2 (q%2), +MT/2)
  //   operand reads of the NEXT phase: activation tiles [MT/4 q, +MT/4)
  //   finish + fetch of code bytes 2(q%2), 2(q%2)+1 of weight tile q/2 (finish: previous fetch -> wf_next)
  //   up to two direct-to-LDS loads of batch `b` (slots d0, d0+1)
  // and the scheduler is asked to alternate MFMA / VALU / LDS inside the quarter.
  auto phase = [&](const bf16x8_t (&xf_use)[MT], const u32x4_t (&wf_use)[NT], bf16x8_t (&xf_next)[MT], int st_next, int ks_next,
                   u32x4_t (&wf_next)[NT], int sw_fin, int ks_fin, int ks_fetch, const BatchAddr& b,
                   int d_first, int d_per_quarter_even, int d_per_quarter_odd) {
    float s8[8];
    load_s8(s8, sw_fin, ks_fin);
    const char* sA = smem + st_next * L::kStageA;
    int d = d_first;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = q >> 1;
      const int nd = (q & 1) ? d_per_quarter_odd : d_per_quarter_even;
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (u < nd) issue_one(b, d + u);
      d += nd;
#pragma unroll
      for (int i = (MT / 4) * q; i < (MT / 4) * (q + 1); ++i)
        xf_next[i] = *reinterpret_cast<const bf16x8_t*>(sA + i * 4096 + x_off[ks_next]);
#pragma unroll
      for (int i = (MT / 2) * (q & 1); i < (MT / 2) * ((q & 1) + 1); ++i)
        acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wf_use[j]), xf_use[i], acc[j][i], 0, 0, 0);
#pragma unroll
      for (int bb = 2 * (q & 1); bb < 2 * (q & 1) + 2; ++bb) {
        finish_byte(wf_next, j, bb, s8);
        fetch_byte(j, ks_fetch, bb);
      }
#pragma unroll
      for (int r = 0; r < MT / 2; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // VALU
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- software pipeline.  Activation tile t lives in A stage t % 4, this wave's codes of k-step t in W stage t % 3.
  // Step t:
  //   phase 0,1 : MFMAs on substeps 0,1 of tile t; batch t+2 is issued, one load per quarter phase
  //   wait for this wave's batch t+1 (batch t+2 stays in flight); barrier: tile t+1 is visible to all waves
  //   phase 2,3 : MFMAs on substeps 2,3; codes of k-step t+1 are read back; phase 3 pre-reads the operands of step t+1
  // That one barrier per step also orders stage reuse: a wave issuing batch t+2 into the A stage of tile t-2 has
  // passed barrier t-1, which every wave reaches only after finishing step t-2.  W stages are wave-private.
  // Weights are expanded just in time: substep ks is fetched two phases and finished one phase before its MFMAs.
  // Global bases of the next batch to issue, carried through the main loop and bumped by a constant per k-step.
  const char *pxb, *pcb, *psb;
  auto seg_base = [&](int q, int step) {
    pxb = reinterpret_cast<const char*>(sg.X[q]) + ((int64_t)step << 7);
    pcb = reinterpret_cast<const char*>(sg.codes[q]) + ((int64_t)step << 5);
    psb = reinterpret_cast<const char*>(sg.scal[q]) + (int64_t)step * 256;
  };
  {  // segment 0 has at least two k-steps (the host puts the widest first): batches 0 and 1 are its
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      seg_base(0, t);
      const BatchAddr bt = batch_addr_at(pxb, pcb, psb, t, t);
#pragma unroll
      for (int d = 0; d < kBatch; ++d) issue_one(bt, d);
    }
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kBatch) : "memory");  // batch 0 landed everywhere, table written
  load_codes(0);
  {
    float s8[8];
    load_s8(s8, 0, 0);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        fetch_byte(j, 0, b);
        finish_byte(wfa, j, b, s8);
        fetch_byte(j, 1, b);
      }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) xfa[i] = *reinterpret_cast<const bf16x8_t*>(smem + i * 4096 + x_off[0]);

  constexpr int kDEven = (kBatch + 7) / 8 > 1 ? 2 : 1;  // loads per even quarter over the 8 quarters of phases 0 and 1
  constexpr int kDOdd = (kBatch - 4 * kDEven + 3) / 4;  // and per odd quarter
  static_assert(4 * kDEven + 4 * kDOdd >= kBatch && kDOdd <= 2 && kDOdd >= 0, "batch does not fit the 8 quarter phases");
  int a0 = 0, w0 = 0;  // A / W stage of the k-step being multiplied
  // One k-step: multiplies tile kt, issues batch kt + 2 from the carried bases, then moves them on by `adv` k-steps
  // (0 past the end of the contraction: the last tile is reloaded, never consumed).
  auto k_step = [&](int64_t adv) {
    const int a1 = (a0 + 1) & 3, a2 = (a0 + 2) & 3;
    const int w1 = w0 == 2 ? 0 : w0 + 1, w2 = w1 == 2 ? 0 : w1 + 1;
    const BatchAddr b = batch_addr_at(pxb, pcb, psb, a2, w2);
    pxb += adv << 7;
    pcb += adv << 5;
    psb += adv * 256;
    phase(xfa, wfa, xfb, a0, 1, wfb, w0, 1, 2, b, 0, kDEven, kDOdd);
    phase(xfb, wfb, xfa, a0, 2, wfa, w0, 2, 3, b, 2 * (kDEven + kDOdd), kDEven, kDOdd);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kBatch) : "memory");
    load_codes(w1);
    phase(xfa, wfa, xfb, a0, 3, wfb, w0, 3, 0, b, kBatch, 0, 0);
    phase(xfb, wfb, xfa, a1, 0, wfa, w1, 0, 1, b, kBatch, 0, 0);
    a0 = a1;
    w0 = w1;
  };
  {
    // The batches are issued segment by segment; inside a segment the lane offsets are loop constants.  The k-steps
    // multiplied meanwhile lag two batches behind and do not care which segment their tile came from.  The last
    // segment runs the two extra steps that drain the pipeline.
    int issued = 2;  // index of the next batch to issue
    for (int q = 0; q < sg.n; ++q) {
      int steps = sg.Kc[q] >> 6;
      if (q == 0) {
        steps -= 2;
        seg_base(0, nk > 2 ? 2 : 1);
      } else {
        set_offsets(sg.Kc[q]);
        seg_base(q, 0);
      }
      if (q == sg.n - 1) steps += 2;
      for (int it = 0; it < steps; ++it) {
        k_step(issued + 1 < nk ? 1 : 0);
        ++issued;
      }
    }
  }

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the clamped batches issued by the last two steps
  // ---- adapter: R extra contraction steps, operands straight from global memory
  //      (one adapter per segment)
  for (int ad = 0; ad < sg.n; ++ad) {
    const uint16_t* __restrict__ lX = sg.lX[ad];
    const uint16_t* __restrict__ lW = sg.lW[ad];
    const int R = sg.R[ad];
    if (!(R > 0 && lX != nullptr)) continue;
    for (int rc = 0; rc < R; rc += 16) {
      const int r0 = rc + 8 * h;
      const bool in = r0 < R;  // R % 8 == 0: a lane's 8 indices are all in or all out
      bf16x8_t wfr[NT], xfr[MT];
      // every request of the step first, then their uses: one trip to memory per step (with the scaling between two
      // loads the compiler waited for each of them in turn)
      u32x4_t xraw[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        int row = m0 + 32 * i + l31;
        row = row < g.M ? row : g.M - 1;
        xraw[i] = u32x4_t{0, 0, 0, 0};
        if (in) xraw[i] = *reinterpret_cast<const u32x4_t*>(lX + (int64_t)row * g.ldlx + r0);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        int col = n0 + wv * 64 + 32 * j + l31;
        col = col < g.Nout ? col : g.Nout - 1;
        u32x4_t raw = {0, 0, 0, 0};
        if (in) {
          uint32_t e[8];
#pragma unroll
          for (int d = 0; d < 8; ++d) e[d] = lW[(int64_t)(r0 + d) * g.Nout + col];
#pragma unroll
          for (int d = 0; d < 4; ++d) raw[d] = e[2 * d] | (e[2 * d + 1] << 16);
        }
        wfr[j] = __builtin_bit_cast(bf16x8_t, raw);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        u32x4_t raw = xraw[i];
        xfr[i] = __builtin_bit_cast(bf16x8_t, raw);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wfr[j], xfr[i], acc[j][i], 0, 0, 0);
    }
  }

  // ---- epilogue.  acc[j][i][v] = C[m][n] with m = m0 + 32 i + l31 and n = n0 + 64 wv + 32 j + 8 (v/4) + 4 h + v%4.
  //      Stored straight from these registers a wave would write 16-byte pieces of 32 different rows per instruction,
  //      which the memory system turns into partial-line read-modify-writes.  Instead each wave transposes its
  //      BM x 64 band through LDS (the activation ring is free now: BM x 128 bytes per wave) and writes whole
  //      128-byte row segments.  16-byte chunk c of row r sits in slot c ^ (r & 7): both sides are conflict-free.
  __syncthreads();  // every wave is done reading the activation ring
  if (n0 + wv * 64 >= g.Nout) return;  // the whole 64-column band of this wave lies outside (no barrier follows)
  {
    char* band = smem + wv * (BM * 128);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const int r = 32 * i + l31;
          u32x2_t o;
          o.x = pack_bf16x2(acc[j][i][4 * q + 0], acc[j][i][4 * q + 1]);
          o.y = pack_bf16x2(acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]);
          *reinterpret_cast<u32x2_t*>(band + r * 128 + (((4 * j + q) ^ (r & 7)) << 4) + 8 * h) = o;
        }
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int c = lane & 7;
    uint16_t* crow = g.C + n0 + wv * 64 + 8 * c;
#pragma unroll 8
    for (int t = 0; t < 4 * MT; ++t) {
      const int r = 8 * t + (lane >> 3);
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(band + r * 128 + ((c ^ (r & 7)) << 4));
      if (m0 + r < g.M) *reinterpret_cast<u32x4_t*>(crow + (int64_t)(m0 + r) * g.Nout) = v;
    }
  }
#endif
}

// C[m][n] = bf16((sum over slices of part[s][m][n] + bias[n]) * cscale[n]); a thread takes 8 consecutive columns, those from
// element e on; mn = M * Nout elements per slice.
__device__ __forceinline__ void sum_slices(int64_t e, const float* __restrict__ part, int splits, int64_t mn, int Nout,
                                           const uint16_t* __restrict__ bias, const uint16_t* __restrict__ cscale, uint16_t* __restrict__ C) {
  float v[8];
  {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(part + e), b = *reinterpret_cast<const f32x4_t*>(part + e + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
  for (int sidx = 1; sidx < splits; ++sidx) {
    const float* p = part + (int64_t)sidx * mn + e;
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p), b = *reinterpret_cast<const f32x4_t*>(p + 4);
    v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w; v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
  }
  const int n = (int)(e % Nout);  // Nout % 8 == 0: the 8 columns share a row
  if (bias) {
    const u32x4_t bb = *reinterpret_cast<const u32x4_t*>(bias + n);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      v[2 * d] += bits_f32(bb[d] << 16);
      v[2 * d + 1] += bits_f32(bb[d] & 0xffff0000u);
    }
  }
  if (cscale) {
    const u32x4_t cc = *reinterpret_cast<const u32x4_t*>(cscale + n);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      v[2 * d] *= bits_f32(cc[d] << 16);
      v[2 * d + 1] *= bits_f32(cc[d] & 0xffff0000u);
    }
  }
  u32x4_t o;
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] = pack_bf16x2(v[2 * d], v[2 * d + 1]);
  *reinterpret_cast<u32x4_t*>(C + e) = o;
}

constexpr int kReduceElements = 256 * 8;  // of a workgroup

// A launch of 5 - 6 us, half of it the way to the first load, which a choice among outputs lengthens (33 x 1024 in sixteen slices
// 6.7 us when every thread looked its output up, 6.1 as it is): one output's sum takes its arguments as they are ...
__global__ __launch_bounds__(256) void nf4_gemm_rs_reduce_kernel(const float* __restrict__ part, int splits, int64_t mn, int Nout,
                                                                 const uint16_t* __restrict__ bias, const uint16_t* __restrict__ cscale,
                                                                 uint16_t* __restrict__ C) {
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (e < mn) sum_slices(e, part, splits, mn, Nout, bias, cscale, C);
}

// ... and those of a group find theirs once per workgroup: output q is the business of the workgroups [wg_end[q - 1], wg_end[q]).
struct RsReduce {
  const float* part[kGroupMax];
  const uint16_t* bias[kGroupMax];
  uint16_t* C[kGroupMax];
  int64_t mn[kGroupMax];
  int Nout[kGroupMax], splits[kGroupMax], wg_end[kGroupMax];
};
__global__ __launch_bounds__(256) void nf4_gemm_rs_group_reduce_kernel(const RsReduce r) {
  int q = 0;
  while ((int)blockIdx.x >= r.wg_end[q]) ++q;  // uniform; the grid ends at wg_end[kGroupMax - 1]
  const int wg = (int)blockIdx.x - (q ? r.wg_end[q - 1] : 0);
  const int64_t e = ((int64_t)wg * 256 + threadIdx.x) * 8;
  if (e < r.mn[q]) sum_slices(e, r.part[q], r.splits[q], r.mn[q], r.Nout[q], r.bias[q], nullptr, r.C[q]);
}

int reduce_workgroups(int64_t elements) { return (int)((elements + kReduceElements - 1) / kReduceElements); }

// The sum over `splits` slices into one output
int launch_reduce(const RsArgs& g, int splits, hipStream_t s) {
  const int64_t mn = (int64_t)g.M * g.Nout;
  nf4_gemm_rs_reduce_kernel<<<dim3((unsigned)reduce_workgroups(mn)), dim3(256), 0, s>>>(g.part, splits, mn, g.Nout, g.bias, g.cscale, g.C);
  return check_launch("nf4_gemm_rs_reduce");
}

// the LDS limit is a per-device attribute of the function: set it for the current device once (a race only repeats the call)
int reserve_lds(const void* fn, bool (&set)[64]) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (dev >= 0 && set[dev]) return TTAMD_OK;
  const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, RsLayout::kTotal);
  if (e != hipSuccess) return fail(TTAMD_ELAUNCH, "nf4_gemm_rs: cannot reserve %d bytes of LDS: %s", RsLayout::kTotal, hipGetErrorString(e));
  if (dev >= 0) set[dev] = true;
  return TTAMD_OK;
}
dim3 wide_grid(RsArgs& g) {
  g.tiles_m = (g.M + kBM - 1) / kBM;
  g.tiles_n = (g.Nout + kBN - 1) / kBN;
  return dim3((unsigned)(g.tiles_m * g.tiles_n));
}
template <int MODE>
int launch_rs16(RsArgs& g, hipStream_t s) {
  static bool set[64] = {};
  if (int rc = reserve_lds(reinterpret_cast<const void*>(&nf4_gemm_rs16_kernel<MODE>), set)) return rc;
  const dim3 grid = wide_grid(g);
  nf4_gemm_rs16_kernel<MODE><<<grid, dim3(256), RsLayout::kTotal, s>>>(g);
  return check_launch("nf4_gemm_rs");
}
int launch_segments(RsArgs& g, const RsSegs& sg, hipStream_t s) {
  static bool set[64] = {};
  if (int rc = reserve_lds(reinterpret_cast<const void*>(&nf4_gemm_rs_segments_kernel), set)) return rc;
  const dim3 grid = wide_grid(g);
  nf4_gemm_rs_segments_kernel<<<grid, dim3(256), RsLayout::kTotal, s>>>(g, sg);
  return check_launch("nf4_gemm_rs");
}

size_t slabs_bytes(int slabs, int64_t M, int64_t Nout) { return slabs > 1 ? (size_t)slabs * (size_t)M * (size_t)Nout * sizeof(float) : 0; }

// Whether a product of one chain of sums per output (nmid_min_chains) takes 256-row tiles: where they cost less than 1 / 0.95 of
// nf4_gemm_mid_kernel's way.  Time in us by rounds of the 256 CUs and 64-wide steps, fitted to products of 600 - 2047 rows: 14336 x
// 4096 at 1000 tokens 108 against 124 on tiles of 128 rows, at 1500 (a second, part-filled round) 204 against 192; grad-input of
// 4096 x 14336 at 900 112 and 127.
// A 256-row tile adds the whole contraction in one chain, the other tiles' wave groups half of it each.  The longer chain is
// admitted only where 256-row tiles take fewer than 5/9 of the rounds of 128-row ones (a round of theirs costs 1.8): beyond, at more
// than 16384 outputs, it gained 1 - 5 % (28672 x 8192 at 1200 tokens 609 -> 581 us) and had 1.5 times the rounding error.
bool wide_tiles_pay(int64_t M, int64_t Nout, int64_t Kc, double mid_cost) {
  if (nmid_min_chains(M, Nout, Kc) > 1) return false;
  const int64_t tiles_n = (Nout + kBN - 1) / kBN, tiles = ((M + 255) / 256) * tiles_n;
  const int64_t rounds = (tiles + 255) / 256, rounds128 = (((M + 127) / 128) * tiles_n + 255) / 256;
  if (9 * rounds >= 5 * rounds128) return false;
  const double k = (double)(Kc / 64), r = (double)rounds;
  const double wide = 2.4 + 13.0 * r + k * (1.07 * r + 0.47 * (double)tiles / 256);
  return mid_cost > 0.95 * wide;
}

// A product that is neither a few tokens' nor on the expanded weight
GemmPlan fused_plan(int64_t M, int64_t Nout, int64_t Kc, size_t scratch, bool forward) {
  GemmPlan f = {};
  for (bool may_slice = true;; may_slice = false) {  // an unsliced plan of the first needs no memory
    double cost;
    f.mid = nmid_plan(M, Nout, Kc, may_slice, true, forward, &cost);
    f.wide = wide_tiles_pay(M, Nout, Kc, cost);
    if (f.wide) f.mid.slices = 1;
    f.bytes = slabs_bytes(f.mid.slices, M, Nout);
    if (f.bytes <= scratch) return f;
  }
}

}  // namespace

GemmPlan plan_gemm_rs(int64_t M, int64_t Nout, int64_t Kc, size_t scratch, bool forward) {
  GemmPlan p = {};
  p.bytes = dense_workspace_bytes(M, Nout, Kc);
  p.dense = p.bytes > 0 && scratch >= p.bytes;
  return p.dense ? p : fused_plan(M, Nout, Kc, scratch, forward);
}

// The expanded weight, or the slabs of the plan with the most of them, and at least as many as the contraction has chains of sums,
// also where the plan keeps those in registers.
size_t gemm_rs_workspace_bytes(int64_t M, int64_t Nout, int64_t Kc) {
  if (const size_t dense = dense_workspace_bytes(M, Nout, Kc)) return dense;
  int slabs = nmid_min_chains(M, Nout, Kc);
  for (const bool forward : {false, true}) {
    if (forward && Nout < 2 * Kc) break;  // the same plan
    const int n = fused_plan(M, Nout, Kc, kAnyScratch, forward).mid.slices;
    slabs = n > slabs ? n : slabs;
  }
  return slabs_bytes(slabs, M, Nout);
}

// Up to 16 tokens, and up to 64 where that kernel is the faster or the tiles would not cut the contraction
bool few_tokens(int64_t M, int64_t Nout, int64_t Kc) {
  return small_m_applies(M, Nout, Kc, true) || (M <= small_m_limit() && gemm_rs_workspace_bytes(M, Nout, Kc) == 0);
}

extern "C" int ttamd_nf4_gemm_plan(int64_t M, int64_t n_out, int64_t k_contract, int may_slice, int by_128, int forward, int* tile_rows, int* slices, int* chain) {
  TT_REQUIRE(M > 0 && n_out > 0 && k_contract > 0 && n_out % 64 == 0 && k_contract % 64 == 0 && tile_rows && slices && chain, "nf4_gemm_plan: bad argument");
  if (dense_path_applies(M, n_out, k_contract)) return fail(TTAMD_EUNSUPPORTED, "nf4_gemm_plan: a product on the expanded weight");
  GemmPlan f = {};
  double cost;
  if (by_128) {
    f = fused_plan(M, n_out, k_contract, may_slice ? kAnyScratch : 0, forward != 0);
  } else {  // as plan_gemm_rs_group_dx
    f.mid = nmid_plan(M, n_out, k_contract, true, false, forward != 0, &cost);
    if (!may_slice && f.mid.slices > 1) f.mid = nmid_plan(M, n_out, k_contract, false, false, forward != 0, &cost);
  }
  const NMidPlan& p = f.mid;
  *tile_rows = f.wide ? 256 : p.rows;
  *slices = p.slices;
  *chain = f.wide ? (int)k_contract : 32 * (p.chain > 0 && p.chain < p.steps ? p.chain : p.steps);
  return TTAMD_OK;
}

// The rows of the adapter activation lX are ldlx elements apart (a group keeps its members' activations side by side).
int run_gemm_rs(const void* X, const uint8_t* codes, const void* scal, int mode, const void* lX, int ldlx, const void* lW,
                bool lw_row_major, int R, float lscale, const void* bias, const void* cscale, void* C, int64_t M, int64_t Nout,
                int64_t Kc, const GemmPlan& p, void* workspace, hipStream_t s) {
  // per-lane byte offsets inside the kernel are 32-bit: the weight must fit them, and a token dimension too long for
  // them is cut into row ranges (multiples of the 256-row tile) that are launched one after the other
  TT_REQUIRE(Nout * Kc / 2 < (int64_t(1) << 32) && Nout * (Kc / 64) * 4 < (int64_t(1) << 32) && Kc * 2 * 256 < (int64_t(1) << 32),
             "nf4_gemm: weight too large for 32-bit offsets (Nout=%lld Kc=%lld)", (long long)Nout, (long long)Kc);
  const int64_t max_rows = (((int64_t(1) << 32) - 1) / (Kc * 2)) / 256 * 256;
  if (M > max_rows) {
    for (int64_t r0 = 0; r0 < M; r0 += max_rows) {
      const int64_t rows = M - r0 < max_rows ? M - r0 : max_rows;
      const int rc = run_gemm_rs(reinterpret_cast<const uint16_t*>(X) + r0 * Kc, codes, scal, mode,
                                 lX ? reinterpret_cast<const uint16_t*>(lX) + r0 * ldlx : nullptr, ldlx, lW, lw_row_major, R, lscale, bias,
                                 cscale, reinterpret_cast<uint16_t*>(C) + r0 * Nout, rows, Nout, Kc,
                                 plan_gemm_rs(rows, Nout, Kc, 0, mode != 1), nullptr, s);
      if (rc != TTAMD_OK) return rc;
    }
    return TTAMD_OK;
  }
  // many tokens and room for the expanded weight: expand once, then the plain bf16 GEMM
  if (p.dense)
    return run_gemm_dense(X, codes, scal, mode, lX, ldlx, lW, lw_row_major, R, lscale, bias, cscale, C, M, Nout, Kc, workspace, s);
  RsArgs g = {};
  g.X = reinterpret_cast<const uint16_t*>(X);
  g.codes = codes;
  g.scal = reinterpret_cast<const float*>(scal);
  g.lX = reinterpret_cast<const uint16_t*>(lX);
  g.lW = reinterpret_cast<const uint16_t*>(lW);
  g.bias = reinterpret_cast<const uint16_t*>(bias);
  g.cscale = reinterpret_cast<const uint16_t*>(cscale);
  g.C = reinterpret_cast<uint16_t*>(C);
  g.M = (int)M; g.Nout = (int)Nout; g.Kc = (int)Kc; g.R = R;
  g.lw_row_major = lw_row_major ? 1 : 0;
  g.ldlx = ldlx;
  g.lscale = lscale;
  if (p.wide) return mode == 1 ? launch_rs16<1>(g, s) : mode == 2 ? launch_rs16<2>(g, s) : launch_rs16<0>(g, s);
  const int slices = p.mid.slices;
  TT_REQUIRE(slices == 1 || aligned16(workspace), "nf4_gemm: workspace must be 16-byte aligned");
  g.part = slices > 1 ? reinterpret_cast<float*>(workspace) : nullptr;
  const int rc = run_nf4_gemm_mid(mode, g, p.mid, nullptr, nullptr, s);
  return rc != TTAMD_OK || slices == 1 ? rc : launch_reduce(g, slices, s);
}

// The grouped grad-input's plan: one contraction over the members' columns (steps of 128 only where each is whole steps).
GemmPlan plan_gemm_rs_group_dx(const GroupDx& d, size_t scratch) {
  int64_t n_total = 0;
  bool by_128 = true;
  for (int i = 0; i < d.n; ++i) {
    n_total += d.N[i];
    by_128 = by_128 && d.N[i] % 128 == 0;
  }
  GemmPlan p = {};
  for (bool may_slice = true;; may_slice = false) {
    double cost;
    p.mid = nmid_plan(d.M, d.K, n_total, may_slice, by_128, false, &cost);
    p.wide = p.mid.slices == 1 && ((d.M + kBM - 1) / kBM) * ((d.K + kBN - 1) / kBN) >= 256;
    p.bytes = slabs_bytes(p.mid.slices, d.M, d.K);
    if (p.bytes <= scratch) return p;
  }
}

// Where nf4_gemm_mid_kernel serves the members' forwards, those on 64-row tiles share a launch and the others one, each
// member with the slices and chains of a launch of its own (the same bits).  Launches of their own leave CUs idle and end in a
// sum each: 4096 + 1024 + 1024 rows of 4096 at 333 tokens 63 us apart, 44 here.  Without memory for the slices every member is
// planned as a call of its own without a workspace.
GroupFwdPlan plan_gemm_rs_group_fwd(const GroupGemm& d, bool room) {
  GroupFwdPlan g = {};
  g.one_launch = d.n >= 2 && d.M * d.K * 2 < (int64_t(1) << 32) && d.K * 2 * 256 < (int64_t(1) << 32);
  size_t sum = 0, most = 0;
  for (int i = 0; i < d.n; ++i) {
    const GemmPlan& p = g.member[i] = plan_gemm_rs(d.M, d.N[i], d.K, room ? kAnyScratch : 0, true);
    g.one_launch = g.one_launch && d.bscal_t[i] && d.N[i] * d.K / 2 < (int64_t(1) << 32) && !p.wide && !dense_path_applies(d.M, d.N[i], d.K);
    sum += p.bytes;
    most = p.bytes > most ? p.bytes : most;
  }
  g.bytes = g.one_launch ? sum : most;
  return g;
}

int run_gemm_rs_group_fwd(const void* x, const GroupGemm& d, const void* h_cat, const GroupFwdPlan& gp, void* workspace, hipStream_t s) {
  TT_REQUIRE(aligned16(workspace), "nf4_lora_group_fwd: workspace must be 16-byte aligned");
  if (!gp.one_launch) {
    for (int i = 0; i < d.n; ++i) {
      const void* sc = d.bscal_t[i] ? d.bscal_t[i] : d.bscal[i];
      if (int rc = run_gemm_rs(x, d.codes[i], sc, d.bscal_t[i] ? 2 : 0, reinterpret_cast<const uint16_t*>(h_cat) + d.r_off[i], d.r_off[d.n],
                               d.lora_b[i], true, d.rank[i], d.scale[i], d.bias[i], nullptr, d.y[i], d.M, d.N[i], d.K, gp.member[i], workspace, s))
        return rc;
    }
    return TTAMD_OK;
  }
  NMidPlan p[kGroupMax];
  for (int i = 0; i < d.n; ++i) p[i] = gp.member[i].mid;
  RsReduce r = {};
  int64_t part = 0;
  int sum_wgs = 0, sums = 0;
  for (const bool small : {false, true}) {
    int64_t widths[kGroupMax];
    NMidPlan plans[kGroupMax];
    int who[kGroupMax], n = 0;
    for (int i = 0; i < d.n; ++i)
      if ((p[i].rows == 64) == small) {
        widths[n] = d.N[i];
        plans[n] = p[i];
        who[n++] = i;
      }
    if (n == 0) continue;
    RsMembers m = {};
    RsArgs g = {};
    g.X = reinterpret_cast<const uint16_t*>(x);
    g.M = (int)d.M;
    g.Kc = (int)d.K;
    g.lw_row_major = 1;
    g.ldlx = d.r_off[d.n];
    g.part = reinterpret_cast<float*>(workspace);
    m.n = n;
    NMidPlan all = plans[0];
    all.rows = nmid_group_rows(d.M, widths, plans, n);
    const int cols = nmid_cols(all.rows);
    int slots = 0;
    for (int k = 0; k < n; ++k) {
      const int i = who[k];
      m.codes[k] = d.codes[i];
      m.scal[k] = d.bscal_t[i];
      m.lX[k] = reinterpret_cast<const uint16_t*>(h_cat) + d.r_off[i];
      m.lW[k] = d.lora_b[i];
      m.bias[k] = d.bias[i];
      m.C[k] = d.y[i];
      m.Nout[k] = (int)d.N[i];
      m.R[k] = d.rank[i];
      m.lscale[k] = d.scale[i];
      m.steps[k] = plans[k].steps;
      m.slices[k] = plans[k].slices;
      m.chain[k] = plans[k].chain > 0 ? plans[k].chain : plans[k].steps + 1;  // a chain longer than the slice never ends in it
      all.chain = plans[k].chain > all.chain ? plans[k].chain : all.chain;
      slots += ((int)(((d.M + all.rows - 1) / all.rows) * ((d.N[i] + cols - 1) / cols)) * plans[k].slices + 7) / 8;
      m.slot_end[k] = slots;
      m.part_at[k] = part;
      if (plans[k].slices > 1) {
        const int64_t mn = d.M * d.N[i];
        r.part[sums] = g.part + part;
        r.bias[sums] = d.bias[i];
        r.C[sums] = d.y[i];
        r.mn[sums] = mn;
        r.Nout[sums] = (int)d.N[i];
        r.splits[sums] = plans[k].slices;
        sum_wgs += reduce_workgroups(mn);
        r.wg_end[sums++] = sum_wgs;
        part += mn * plans[k].slices;
      }
    }
    if (int rc = run_nf4_gemm_mid(2, g, all, nullptr, &m, s)) return rc;
  }
  if (sums == 0) return TTAMD_OK;
  nf4_gemm_rs_group_reduce_kernel<<<dim3((unsigned)sum_wgs), dim3(256), 0, s>>>(r);
  return check_launch("nf4_gemm_rs_reduce");
}

// Grad-input of a group of layers with a common input, as one GEMM over the concatenated contraction:
//   gx[M, K] = sum_i gy_i[M, N_i] . D(W_i)[N_i, K] + gh_i[M, R_i] . A_i[R_i, K]
// with the members' transposed copies (codes [K, N_i / 2], per-element scalers [K / 64, N_i]); gh_i = columns
// [r_off[i], r_off[i + 1]) of gh_cat.  The sum over members is taken in fp32, before the one rounding to bf16.
// A launch of few tiles is sliced like a single layer's where there is memory for it: unsliced it
// takes its 256 - 448 k-steps however few workgroups there are.  Unsliced -> sliced, us: 14336 + 14336 rows of 4096 at 100
// tokens 287 -> 49, at 333 293 -> 111, at 1000 302 -> 246; 4096 + 1024 + 1024 at 333 67 -> 38, at 1000 75 -> 70; 8192 + 8192
// rows of 2048 at 333 164 -> 45.
int run_gemm_rs_group_dx(const GroupDx& d, const void* gh_cat, void* gx, const GemmPlan& p, void* workspace, hipStream_t s) {
  TT_REQUIRE(d.n >= 1 && d.n <= kGroupMax, "nf4_group_dx: %d members", d.n);
  RsSegs sg = {};
  sg.n = d.n;
  int64_t max_n = 0;
  int first = 0;  // the widest member goes first: the kernel takes its first two batches from segment 0
  for (int i = 0; i < d.n; ++i) {
    TT_REQUIRE(d.N[i] > 0 && d.N[i] % 64 == 0, "nf4_group_dx: N (%lld) must be a positive multiple of 64", (long long)d.N[i]);
    TT_REQUIRE(aligned16(d.gy[i]) && aligned16(d.codes_t[i]) && aligned16(d.scal_t[i]), "nf4_group_dx: pointers must be 16-byte aligned");
    if (d.N[i] > max_n) {
      max_n = d.N[i];
      first = i;
    }
  }
  if (max_n < 128) return fail(TTAMD_EUNSUPPORTED, "nf4_group_dx: the widest member must have at least 128 outputs (has %lld)", (long long)max_n);
  for (int k = 0; k < d.n; ++k) {
    const int i = k == 0 ? first : (k <= first ? k - 1 : k);  // first, then the others in their order
    sg.X[k] = d.gy[i];
    sg.codes[k] = d.codes_t[i];
    sg.scal[k] = d.scal_t[i];
    sg.lX[k] = d.rank[i] > 0 ? reinterpret_cast<const uint16_t*>(gh_cat) + d.r_off[i] : nullptr;
    sg.lW[k] = d.lora_a[i];
    sg.Kc[k] = (int)d.N[i];
    sg.R[k] = d.rank[i];
  }
  // per-lane byte offsets inside the kernel are 32-bit
  if (!(d.K * max_n / 2 < (int64_t(1) << 32) && d.K / 64 * max_n * 4 < (int64_t(1) << 32) && d.M * max_n * 2 < (int64_t(1) << 32)))
    return fail(TTAMD_EUNSUPPORTED, "nf4_group_dx: operands too large for 32-bit offsets (M=%lld K=%lld N=%lld)", (long long)d.M,
                (long long)d.K, (long long)max_n);
  RsArgs g = {};
  g.C = reinterpret_cast<uint16_t*>(gx);
  g.M = (int)d.M; g.Nout = (int)d.K;
  g.lw_row_major = 0;
  g.ldlx = d.r_off[d.n];
  g.lscale = 1.0f;
  if (p.wide) return launch_segments(g, sg, s);
  TT_REQUIRE(p.mid.slices == 1 || aligned16(workspace), "nf4_group_dx: workspace must be 16-byte aligned");
  g.part = reinterpret_cast<float*>(workspace);
  const int rc = run_nf4_gemm_mid(1, g, p.mid, &sg, nullptr, s);
  return rc != TTAMD_OK || p.mid.slices == 1 ? rc : launch_reduce(g, p.mid.slices, s);
}

}  // namespace ttamd
