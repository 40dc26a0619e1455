// Arguments of the fused NF4 GEMMs (nf4_gemm_rs.hip, nf4_gemm_mid.hip).
#pragma once
#include "common.h"
#include "group.h"

namespace ttamd {

struct RsArgs {
  const uint16_t* X;     // [M, Kc] bf16 activations
  const uint8_t* codes;  // [Nout, Kc/2] packed NF4 codes of the weight view
  const float* scal;     // block scalers, fp32: MODE 0 [Nout, Kc/64]; MODE 2 [Kc/64, Nout]; MODE 1 per element [Nout/64, Kc]
  const uint16_t* lX;    // adapter activations [M, R] bf16 (rows ldlx elements apart) or null
  const uint16_t* lW;    // adapter weights: [Nout, R] (lw_row_major) or [R, Nout] bf16, or null
  const uint16_t* bias;  // [Nout] bf16 or null
  const uint16_t* cscale;  // [Nout] bf16 or null: C = (acc + bias) * cscale per column (DoRA's magnitude / norm)
  uint16_t* C;           // [M, Nout] bf16
  float* part;           // slices: fp32 partial products [slices, M, Nout], added up by a launch of their own
  int M, Nout, Kc, R;
  int lw_row_major;
  int ldlx;
  float lscale;
  int tiles_m, tiles_n;
  // nf4_gemm_mid_kernel
  int slices, steps;   // slices of a tile's contraction, steps of one
  int chain;           // steps of a chain of sums
  int items, per_xcd;  // workgroups of the launch, of an XCD
};

// The contraction is the concatenation of up to kGroupMax segments, each with its own activation, weight
// view and adapter (the grad-input of a group of layers with a common input: gx = sum_i gy_i . D(W_i) + gh_i . A_i is
// one GEMM whose contraction runs over the members' output columns one member after the other).  g.X / codes / scal /
// Kc / lX / lW / R are then unused; M, Nout, C and ldlx are shared.
struct RsSegs {
  const uint16_t* X[kGroupMax];     // [M, Kc[i]]
  const uint8_t* codes[kGroupMax];  // [Nout, Kc[i] / 2]
  const float* scal[kGroupMax];     // MODE 1: [Nout / 64, Kc[i]]
  const uint16_t* lX[kGroupMax];    // adapter activations, rows g.ldlx apart, or null
  const uint16_t* lW[kGroupMax];    // adapter weights [R[i], Nout]
  int Kc[kGroupMax], R[kGroupMax];
  int n;
};

// The forwards of layers with a common input X as one launch.  Member q has the workgroups [slot_end[q - 1], slot_end[q]) of
// every XCD: its tiles in the slices a launch of its own has (the same bits), its partial products [slices, M, Nout[q]] at part_at[q].
// g.codes / scal / lX / lW / R / lscale / bias / C / Nout / steps / slices / chain are then unused, MODE is 2.
struct RsMembers {
  const uint8_t* codes[kGroupMax];
  const float* scal[kGroupMax];
  const uint16_t* lX[kGroupMax];
  const uint16_t* lW[kGroupMax];
  const uint16_t* bias[kGroupMax];
  uint16_t* C[kGroupMax];
  int64_t part_at[kGroupMax];
  int Nout[kGroupMax], R[kGroupMax], slot_end[kGroupMax], steps[kGroupMax], slices[kGroupMax], chain[kGroupMax];
  float lscale[kGroupMax];
  int n;
};

int nmid_cols(int rows);
// the chains of sums that an output's contraction has at least
int nmid_min_chains(int64_t M, int64_t Nout, int64_t Kc);
// The plan of least time; *cost: its time in us by the model.  may_slice: there is memory for slices; by_128: the contraction may
// be taken 128 indices at a time (every segment of it is a multiple).
NMidPlan nmid_plan(int64_t M, int64_t Nout, int64_t Kc, bool may_slice, bool by_128, bool forward, double* cost);
// Tile rows of one launch for n members with plans of 64 rows, or of 96 and 128: those give an output the same bits.
int nmid_group_rows(int64_t M, const int64_t* Nout, const NMidPlan* p, int n);
// mode 0, 1, 2: scaler modes of RsArgs; segs (mode 1) or members (mode 2) or neither.  With slices (p.slices > 1, or a member's)
// g.part receives the partial products.
int run_nf4_gemm_mid(int mode, RsArgs& g, const NMidPlan& p, const RsSegs* segs, const RsMembers* members, hipStream_t s);

}  // namespace ttamd
