// Internal interface between the translation units that serve a group of LoRA linears with a common input
// (q/k/v of torchtune/modules/attention.py:234,262-263; gate/up of torchtune/modules/feed_forward.py:50-53).
#pragma once
#include "common.h"

namespace ttamd {

constexpr int kGroupMax = TTAMD_GROUP_MAX;  // most members of a group

// What the rank-r products need to know about a group.  The members' hidden activations lie side by side in one
// [M, r_off[n]] tensor (member i in columns [r_off[i], r_off[i + 1])), and so do their gradients.
struct GroupSkinny {
  int n;
  int64_t M, K;
  int64_t N[kGroupMax];
  int rank[kGroupMax], r_off[kGroupMax + 1];
  float scale[kGroupMax];
  const uint16_t* lora_a[kGroupMax];  // [rank, K]
  const uint16_t* lora_b[kGroupMax];  // [N, rank]
  const uint16_t* gy[kGroupMax];      // [M, N]        (backward)
  uint16_t* ga[kGroupMax];            // [rank, K] out (backward)
  uint16_t* gb[kGroupMax];            // [N, rank] out (backward)
};

// What the fused NF4 GEMMs need to know about a group (forward).
struct GroupGemm {
  int n;
  int64_t M, K;
  int64_t N[kGroupMax];
  int rank[kGroupMax], r_off[kGroupMax + 1];
  float scale[kGroupMax];
  const uint8_t* codes[kGroupMax];    // [N, K/2]
  const float* bscal[kGroupMax];      // [N, K/64]
  const float* bscal_t[kGroupMax];    // [K/64, N] or null
  const uint16_t* lora_b[kGroupMax];  // [N, rank]
  const uint16_t* bias[kGroupMax];    // [N] or null
  uint16_t* y[kGroupMax];             // [M, N] out
};

// What the grouped grad-input needs (backward): the members' transposed copies and gradients.
struct GroupDx {
  int n;
  int64_t M, K;
  int64_t N[kGroupMax];
  int rank[kGroupMax], r_off[kGroupMax + 1];
  const uint16_t* gy[kGroupMax];       // [M, N]
  const uint8_t* codes_t[kGroupMax];   // [K, N/2] or null (then codes / bscal serve the expanded-weight path)
  const float* scal_t[kGroupMax];      // [K/64, N] or null
  const uint8_t* codes[kGroupMax];     // [N, K/2]
  const float* bscal[kGroupMax];       // [N, K/64]
  const uint16_t* lora_a[kGroupMax];   // [rank, K]
};

// How nf4_gemm_mid_kernel runs a product: tiles of 64 rows x 128 columns (steps of 128 contraction indices), of 96 or of 128 x 256
// (steps of 64); slices of the contraction of `steps` steps each; chain > 0: chains of sums end after so many steps.
struct NMidPlan {
  int rows, slices, steps, chain;
};
// How a product of more than a few tokens runs: on the weight expanded once, on the fused 256-row tiles, or as mid says.  An entry
// point plans once and hands the plan down.
struct GemmPlan {
  bool dense, wide;
  NMidPlan mid;
  size_t bytes;  // of memory that it writes
};
constexpr size_t kAnyScratch = SIZE_MAX;
// nf4_gemm_rs.hip.  scratch: bytes at hand (kAnyScratch: as many as it asks for); forward: else the grad-input
GemmPlan plan_gemm_rs(int64_t M, int64_t Nout, int64_t Kc, size_t scratch, bool forward);
// workspace: p.bytes
int run_gemm_rs(const void* X, const uint8_t* codes, const void* scal, int mode, const void* lX, int ldlx, const void* lW,
                bool lw_row_major, int R, float lscale, const void* bias, const void* cscale, void* C, int64_t M, int64_t Nout,
                int64_t Kc, const GemmPlan& p, void* workspace, hipStream_t s);
// what callers of the per-kernel entry points bring (ttamd_nf4_gemm_workspace_bytes)
size_t gemm_rs_workspace_bytes(int64_t M, int64_t Nout, int64_t Kc);
// the forward of M tokens runs the few-token kernel whatever memory there is
bool few_tokens(int64_t M, int64_t Nout, int64_t Kc);
// The grouped grad-input on the fused tiles
GemmPlan plan_gemm_rs_group_dx(const GroupDx& d, size_t scratch);
int run_gemm_rs_group_dx(const GroupDx& d, const void* gh_cat, void* gx, const GemmPlan& p, void* workspace, hipStream_t s);
// The members' forwards: in one launch or two, or (one_launch false) one after the other in the same memory
struct GroupFwdPlan {
  bool one_launch;
  GemmPlan member[kGroupMax];
  size_t bytes;
};
GroupFwdPlan plan_gemm_rs_group_fwd(const GroupGemm& d, bool room);
int run_gemm_rs_group_fwd(const void* x, const GroupGemm& d, const void* h_cat, const GroupFwdPlan& p, void* workspace, hipStream_t s);

// nf4_gemm.hip: the checked layer calls on a plan of the caller's; plan null: the few-token kernel
int run_lora_linear_fwd(const char* who, const void* x, const uint8_t* quantized_data, const void* block_scalers, const void* block_scalers_t,
                        const void* h, const void* lora_b, int rank, float scale, const void* bias, const void* col_scale, void* y,
                        int64_t M, int64_t N, int64_t K, const GemmPlan* plan, void* workspace, hipStream_t s);
int run_linear_bwd_dx(const void* gy, const uint8_t* quantized_data, const void* block_scalers, const uint8_t* quantized_data_t,
                      const void* block_scalers_t, const void* gh, const void* lora_a, int rank, void* gx, int64_t M, int64_t N,
                      int64_t K, const GemmPlan& plan, void* workspace, hipStream_t s);

// nf4_gemm_dense.hip: expand the weight once into scratch memory, then a plain bf16 GEMM (many tokens)
bool dense_path_applies(int64_t M, int64_t Nout, int64_t Kc);
size_t dense_workspace_bytes(int64_t M, int64_t Nout, int64_t Kc);
// The result taken as the gradient of silu(gate) * up (gate, up [M, Nout] bf16): C receives the gradient of gate, gup
// that of up, and the result itself is not stored.
struct DenseSwigluBwd {
  const void* gate;
  const void* up;
  void* gup;
};
int run_gemm_dense(const void* X, const uint8_t* codes, const void* scal, int mode, const void* lX, int ldlx, const void* lW,
                   bool lw_row_major, int R, float lscale, const void* bias, const void* cscale, void* C, int64_t M, int64_t Nout,
                   int64_t Kc, void* workspace, hipStream_t s, const DenseSwigluBwd* swiglu_bwd = nullptr);
size_t dense_group_fwd_workspace_bytes(const GroupGemm& d);
// act != nullptr: two members of equal width (gate, up); the launch also writes act = silu(y[0]) * y[1]
bool dense_group_gated_applies(const GroupGemm& d);
int run_gemm_dense_group_fwd(const void* x, const GroupGemm& d, const void* h_cat, void* workspace, hipStream_t s, void* act = nullptr,
                             const void* tiles = nullptr);
size_t dense_group_dx_workspace_bytes(const GroupDx& d);
int run_gemm_dense_group_dx(const GroupDx& d, const void* gh_cat, void* gx, void* workspace, hipStream_t s,
                            const void* tiles_fwd = nullptr, bool paired = false);

// C[N, K] = A[M, N]^T . B[M, K], N and K multiples of 64 and any M (gemm_tn.hip); 16-byte aligned operands.
int run_gemm_tn(const void* a, const void* b, void* c, int64_t M, int64_t N, int64_t K, hipStream_t s);
// nf4_small_m.hip: y[i] = x . D(W_i)^T (+ bias) + scale . h_i . lora_b[i]^T for a handful of tokens
int small_m_limit();
// the forward of M tokens on an [N, K] weight runs the few-token kernel (sliced_ok: the tiled kernel may cut its contraction)
bool small_m_applies(int64_t M, int64_t N, int64_t K, bool sliced_ok);
int run_small_m_group(const void* x, const GroupGemm& g, const void* h_cat, void* act, bool* act_done, hipStream_t s);
// the same with h_i = x . lora_a[i]^T formed inside the launches (gated: two members of equal width, act is written too), the
// same bits, where that is the better way; h_cat receives it, or is null
bool few_forms_hidden(const GroupGemm& g, bool gated);
int run_few_with_hidden(const void* x, const GroupGemm& g, const uint16_t* const* lora_a, void* h_cat, void* act, hipStream_t s);

// lora_skinny.hip
size_t group_hidden_ws_bytes(int64_t M, int64_t K, int r_total);
// How h = x . lora_a^T of at most 32 tokens is summed over K (by K alone): in `splits` runs of 64-wide chunks, or (0) by the
// sixteen waves of one workgroup
struct HiddenOrder {
  int splits, chunks_per_split;
};
HiddenOrder hidden_order(int64_t K);
// h_cat[:, r_off[i] : r_off[i + 1]] = x . lora_a[i]^T for every member, in one pass over x
int run_group_hidden(const uint16_t* x, const GroupSkinny& g, uint16_t* h_cat, float* ws, hipStream_t s);
size_t group_lora_bwd_ws_bytes(const GroupSkinny& g);
// gh_cat[:, member i] = scale[i] . gy[i] . lora_b[i];  ga[i] = gh_i^T . x (one pass over x for all members);
// gb[i] = scale[i] . gy[i]^T . h_i
// sw (optional; the gate / up pair of a SwiGLU feed-forward): g.gy[0] and g.gy[1] are then OUTPUTS, the gradients of gate
// and up, which this call derives from the gradient of silu(gate) * up first - in the same pass that forms the products
// reading them where that pass exists (two wide members of equal width), otherwise by the stand-alone kernel.
struct SwigluBwdInputs {
  const uint16_t* gact;  // [M, N]
  const uint16_t* gate;  // [M, N]
  const uint16_t* up;    // [M, N]
};
int run_group_lora_bwd(const uint16_t* x, const uint16_t* h_cat, const GroupSkinny& g, uint16_t* gh_cat, float* ws, hipStream_t s,
                       const SwigluBwdInputs* sw = nullptr);

}  // namespace ttamd
