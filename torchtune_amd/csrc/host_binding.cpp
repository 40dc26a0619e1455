// Host path of the small calls: argument checks, output and workspace allocation, autograd bookkeeping and the launches of
// one layer call in native code.
//
// A decoder layer's linears and their neighbours are a few kernels of 3 - 30 us each at few tokens; the Python wrappers
// (ctypes call, tensor checks, torch.autograd.Function) cost 25 - 35 us per op and direction, so those calls were bound
// by the host: a layer of the 8B shape 360 us at one token for 119 us of kernels, a layer of the 1B shape at 700 tokens
// 1214 us forward + backward for 663 us.  The functions here make the same library calls (include/torchtune_amd.h) with the
// same arguments, and the autograd nodes are C++ ones, so that backward runs without the interpreter too.
//
// This extension is the torch side of the C ABI; libtorchtune_amd.so itself stays free of torch types.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <pybind11/stl.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>

#include "../../include/torchtune_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check(int rc, const char* what) {
  if (rc == TTAMD_OK) return;
  if (rc == TTAMD_EINVAL) TORCH_CHECK_VALUE(false, what, ": ", ttamd_last_error());
  TORCH_CHECK(false, what, " failed (code ", rc, "): ", ttamd_last_error());
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

void need_gpu(const Tensor& t, const char* what) {
  TORCH_CHECK(t.is_cuda(), what, ": expected a tensor on an AMD GPU (device 'cuda'), got device '", t.device().str(),
              "'. torchtune_amd computes only through its HIP kernels.");
}

// a contiguous bf16 tensor on the GPU
Tensor bf16(const Tensor& t, const char* what) {
  need_gpu(t, what);
  TORCH_CHECK_TYPE(t.scalar_type() == at::kBFloat16, what, ": expected a bfloat16 tensor, got ", t.scalar_type());
  return t.contiguous();
}

Tensor scratch(size_t bytes, const Tensor& like) {
  return at::empty({(int64_t)(bytes > 16 ? bytes : 16)}, like.options().dtype(at::kByte));
}

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

// True when the call has to be a node: something is differentiated backward, or carries a forward-mode tangent (the node
// then raises: none of them has a forward-mode rule, and a plain call would drop the tangent).
bool wants_grad(std::initializer_list<const Tensor*> ts) {
  const bool grad = at::GradMode::is_enabled();
  for (const Tensor* t : ts)
    if (t->defined() && ((grad && t->requires_grad()) || t->_fw_grad(0).defined())) return true;
  return false;
}

// A tensor the kernels may read in place of torch's own ops: no forward-mode tangent, no function transform's wrapper, no
// subclass with a dispatch of its own, and no dispatch mode that would have seen those ops (a FLOP counter, a selective
// checkpoint's list of what to save).
bool ordinary(const Tensor& t) {
  if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::Functionalize, c10::DispatchKey::Python});
  return !t.key_set().has_any(wrapped) && !t._fw_grad(0).defined();
}

// The kernels that took over from torch's matmul read 16 bytes at a time; a contiguous view may begin anywhere.
Tensor aligned(const Tensor& t) { return !t.defined() || (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0 ? t : t.clone(); }

int64_t last_dim(const Tensor& t, const char* what) {
  const int64_t n = t.size(-1);
  TORCH_CHECK_VALUE(n > 0, what, ": the last dimension is empty");
  return n;
}

// ---------------------------------------------------------------------------------------------------
// RMSNorm
// ---------------------------------------------------------------------------------------------------
struct NormOut {
  Tensor h, y, rstd;
};

NormOut norm_forward(const Tensor& x, const Tensor* residual, const Tensor& scale, double eps) {
  const Tensor xc = bf16(x, "rms_norm_fwd: x"), sc = bf16(scale, "rms_norm_fwd: scale");
  const c10::DeviceGuard guard(xc.device());
  const int64_t D = last_dim(xc, "rms_norm_fwd"), rows = xc.numel() / D;
  TORCH_CHECK_VALUE(sc.numel() == D, "rms_norm_fwd: scale has ", sc.numel(), " elements, the rows ", D);
  NormOut o;
  o.y = at::empty_like(xc);
  o.rstd = at::empty({rows}, xc.options().dtype(at::kFloat));
  if (residual) {
    const Tensor rc = bf16(*residual, "add_rms_norm_fwd: residual");
    TORCH_CHECK_VALUE(rc.sizes() == xc.sizes(), "add_rms_norm_fwd: x ", xc.sizes(), " and residual ", rc.sizes(), " differ in shape");
    o.h = at::empty_like(xc);
    check(ttamd_add_rms_norm_fwd_bf16(xc.data_ptr(), rc.data_ptr(), sc.data_ptr(), (float)eps, o.h.data_ptr(), o.y.data_ptr(),
                                      o.rstd.data_ptr<float>(), rows, D, stream_of(xc)),
          "add_rms_norm_fwd");
  } else {
    check(ttamd_rms_norm_fwd_bf16(xc.data_ptr(), sc.data_ptr(), (float)eps, o.y.data_ptr(), o.rstd.data_ptr<float>(), rows, D, stream_of(xc)),
          "rms_norm_fwd");
  }
  return o;
}

// (gx, gscale or undefined)
std::pair<Tensor, Tensor> norm_backward(const Tensor& gy, const Tensor& x, const Tensor& scale, const Tensor& rstd, bool want_gscale,
                                        const Tensor& g_add) {
  const Tensor gc = bf16(gy, "rms_norm_bwd: gy"), xc = bf16(x, "rms_norm_bwd: x"), sc = bf16(scale, "rms_norm_bwd: scale");
  const c10::DeviceGuard guard(xc.device());
  const int64_t D = last_dim(xc, "rms_norm_bwd"), rows = xc.numel() / D;
  const Tensor ga = g_add.defined() ? bf16(g_add, "rms_norm_bwd: g_add") : Tensor();
  TORCH_CHECK_VALUE(gc.numel() == xc.numel() && (!ga.defined() || ga.numel() == xc.numel()), "rms_norm_bwd: gradients and x differ in size");
  Tensor gx = at::empty_like(xc), gscale, ws;
  size_t bytes = 0;
  if (want_gscale) {
    gscale = at::empty({D}, xc.options());
    bytes = ttamd_rms_norm_bwd_workspace_bytes(D);
    ws = scratch(bytes, xc);
  }
  check(ttamd_rms_norm_bwd_add_bf16(gc.data_ptr(), xc.data_ptr(), sc.data_ptr(), rstd.data_ptr<float>(), ga.defined() ? ga.data_ptr() : nullptr,
                                    gx.data_ptr(), want_gscale ? gscale.data_ptr() : nullptr, rows, D,
                                    want_gscale ? ws.data_ptr() : nullptr, bytes, stream_of(xc)),
        "rms_norm_bwd");
  return {gx, gscale};
}

struct RMSNormFn : torch::autograd::Function<RMSNormFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& scale, double eps) {
    NormOut o = norm_forward(x, nullptr, scale, eps);
    ctx->save_for_backward({x, scale, o.rstd});
    return o.y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto saved = ctx->get_saved_variables();
    auto [gx, gscale] = norm_backward(g[0], saved[0], saved[1], saved[2], ctx->needs_input_grad(1), Tensor());
    return {gx, gscale, Tensor()};
  }
};

Tensor rms_norm(const Tensor& x, const Tensor& scale, double eps) {
  return wants_grad({&x, &scale}) ? RMSNormFn::apply(x, scale, eps) : norm_forward(x, nullptr, scale, eps).y;
}

// (x, residual, scale) -> (h = x + residual, RMSNorm(h)).  Backward: both inputs receive grad h + the gradient of the norm's
// input, summed in the norm's backward pass.
struct AddRMSNormFn : torch::autograd::Function<AddRMSNormFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& residual, const Tensor& scale, double eps) {
    NormOut o = norm_forward(x, &residual, scale, eps);
    ctx->save_for_backward({o.h, scale, o.rstd});
    ctx->set_materialize_grads(false);  // an output nobody used arrives undefined, not as a tensor of zeros
    return {o.h, o.y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[1].defined()) return {g[0], g[0], Tensor(), Tensor()};  // the normalised output went nowhere
    const auto saved = ctx->get_saved_variables();
    auto [gx, gscale] = norm_backward(g[1], saved[0], saved[1], saved[2], ctx->needs_input_grad(2), g[0]);
    return {gx, gx, gscale, Tensor()};
  }
};

std::pair<Tensor, Tensor> add_rms_norm(const Tensor& x, const Tensor& residual, const Tensor& scale, double eps) {
  if (wants_grad({&x, &residual, &scale})) {
    variable_list o = AddRMSNormFn::apply(x, residual, scale, eps);
    return {o[0], o[1]};
  }
  NormOut o = norm_forward(x, &residual, scale, eps);
  return {o.h, o.y};
}

// ---------------------------------------------------------------------------------------------------
// rotary embedding of q / k with the key / value head expansion; SwiGLU gate
// ---------------------------------------------------------------------------------------------------
Tensor rope_cache_arg(const Tensor& cache, int64_t s, int64_t hd, const char* who) {
  need_gpu(cache, who);
  TORCH_CHECK_VALUE(cache.scalar_type() == at::kFloat && cache.dim() >= 2 && cache.numel() >= s * hd && cache.size(-1) == 2 &&
                        cache.size(-2) == hd / 2,
                    who, ": cache must be fp32 [>= ", s, ", ", hd / 2, ", 2], got ", cache.sizes(), " ", cache.scalar_type());
  return cache.contiguous();
}

variable_list qkv_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cache) {
  const Tensor qc = bf16(q, "qkv_rope_repeat: q"), kc = bf16(k, "qkv_rope_repeat: k"), vc = bf16(v, "qkv_rope_repeat: v");
  TORCH_CHECK_VALUE(qc.dim() == 4 && kc.dim() == 4 && vc.sizes() == kc.sizes() && qc.size(0) == kc.size(0) && qc.size(1) == kc.size(1) &&
                        qc.size(3) == kc.size(3),
                    "qkv_rope_repeat: expected [b, s, n_h, h_d] and two [b, s, n_kv, h_d], got ", qc.sizes(), ", ", kc.sizes(), ", ", vc.sizes());
  const int64_t nh = qc.size(2), nkv = kc.size(2), hd = qc.size(3);
  TORCH_CHECK_VALUE(nkv >= 1 && nh % nkv == 0, "qkv_rope_repeat: ", nh, " query heads against ", nkv, " key / value heads");
  const Tensor cc = rope_cache_arg(cache, qc.size(1), hd, "qkv_rope_repeat");
  const c10::DeviceGuard guard(qc.device());
  Tensor qo = at::empty_like(qc), ko = at::empty_like(qc), vo = at::empty_like(qc);
  check(ttamd_qkv_rope_repeat_bf16(qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), cc.data_ptr<float>(), qo.data_ptr(), ko.data_ptr(), vo.data_ptr(),
                                   qc.size(0), qc.size(1), nh, nkv, hd, stream_of(qc)),
        "qkv_rope_repeat");
  return {qo, ko, vo};
}

struct QKVRopeRepeatFn : torch::autograd::Function<QKVRopeRepeatFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cache) {
    ctx->save_for_backward({cache});
    ctx->saved_data["n_kv"] = k.size(2);
    return qkv_forward(q, k, v, cache);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const Tensor a = bf16(g[0], "qkv_rope_repeat_bwd: gq"), b = bf16(g[1], "qkv_rope_repeat_bwd: gk"), c = bf16(g[2], "qkv_rope_repeat_bwd: gv");
    const c10::DeviceGuard guard(a.device());
    const int64_t nkv = ctx->saved_data["n_kv"].toInt();
    const Tensor cc = ctx->get_saved_variables()[0].contiguous();
    Tensor gq = at::empty_like(a), gk = at::empty({a.size(0), a.size(1), nkv, a.size(3)}, a.options()), gv = at::empty_like(gk);
    check(ttamd_qkv_rope_repeat_bwd_bf16(a.data_ptr(), b.data_ptr(), c.data_ptr(), cc.data_ptr<float>(), gq.data_ptr(), gk.data_ptr(),
                                         gv.data_ptr(), a.size(0), a.size(1), a.size(2), nkv, a.size(3), stream_of(a)),
          "qkv_rope_repeat_bwd");
    return {gq, gk, gv, Tensor()};
  }
};

std::tuple<Tensor, Tensor, Tensor> qkv_rope_repeat(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cache) {
  variable_list o = wants_grad({&q, &k, &v}) ? QKVRopeRepeatFn::apply(q, k, v, cache) : qkv_forward(q, k, v, cache);
  return {o[0], o[1], o[2]};
}

Tensor swiglu_forward(const Tensor& gate, const Tensor& up) {
  const Tensor g = bf16(gate, "swiglu_fwd: gate"), u = bf16(up, "swiglu_fwd: up");
  TORCH_CHECK_VALUE(g.sizes() == u.sizes(), "swiglu_fwd: shapes differ: ", g.sizes(), " vs ", u.sizes());
  const c10::DeviceGuard guard(g.device());
  Tensor out = at::empty_like(g);
  check(ttamd_swiglu_fwd_bf16(g.data_ptr(), u.data_ptr(), out.data_ptr(), g.numel(), stream_of(g)), "swiglu_fwd");
  return out;
}

std::pair<Tensor, Tensor> swiglu_backward(const Tensor& gout, const Tensor& gate, const Tensor& up) {
  const Tensor go = bf16(gout, "swiglu_bwd: gout"), g = bf16(gate, "swiglu_bwd: gate"), u = bf16(up, "swiglu_bwd: up");
  TORCH_CHECK_VALUE(go.numel() == g.numel() && u.numel() == g.numel(), "swiglu_bwd: operands differ in size");
  const c10::DeviceGuard guard(g.device());
  Tensor gg = at::empty_like(g), gu = at::empty_like(u);
  check(ttamd_swiglu_bwd_bf16(go.data_ptr(), g.data_ptr(), u.data_ptr(), gg.data_ptr(), gu.data_ptr(), g.numel(), stream_of(g)), "swiglu_bwd");
  return {gg, gu};
}

struct SwiGLUFn : torch::autograd::Function<SwiGLUFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gate, const Tensor& up) {
    ctx->save_for_backward({gate, up});
    return swiglu_forward(gate, up);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto saved = ctx->get_saved_variables();
    auto [gg, gu] = swiglu_backward(g[0], saved[0], saved[1]);
    return {gg, gu};
  }
};

Tensor swiglu(const Tensor& gate, const Tensor& up) {
  return wants_grad({&gate, &up}) ? SwiGLUFn::apply(gate, up) : swiglu_forward(gate, up);
}

// ---------------------------------------------------------------------------------------------------
// LoRA linears over NF4 weights, fewer tokens than the expand-once path takes
// ---------------------------------------------------------------------------------------------------
// The frozen weight's tensors: codes, block scalers and, where a call may need them, the transposed copies, which the node
// keeps as plain references.  The weight they belong to is a saved variable beside them, so that a write to it between
// forward and backward is an error (the copies would no longer be its).
struct Weight {
  Tensor whole, q, scal, q_t, scal_t;
  int64_t N = 0;
};

void check_weight(const Weight& w, int64_t K, const char* what) {
  need_gpu(w.q, what);
  const int64_t n = w.N * K;
  TORCH_CHECK_VALUE(w.q.scalar_type() == at::kByte && w.q.numel() * 2 == n, what, ": quantized_data holds ", w.q.numel() * 2,
                    " codes, the weight is [", w.N, ", ", K, "]");
  TORCH_CHECK_VALUE(w.scal.scalar_type() == at::kFloat && w.scal.numel() * 64 == n, what, ": block_scalers must be float32 with ", n / 64,
                    " elements");
  if (w.q_t.defined())
    TORCH_CHECK_VALUE(w.q_t.scalar_type() == at::kByte && w.q_t.numel() * 2 == n && w.scal_t.scalar_type() == at::kFloat &&
                          w.scal_t.numel() * 64 == n,
                      what, ": the transposed copies do not hold a [", w.N, ", ", K, "] weight");
}

void* opt_ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

std::vector<int64_t> with_last(const Tensor& x, int64_t last) {
  std::vector<int64_t> s = x.sizes().vec();
  s.back() = last;
  return s;
}

struct Member {
  Weight w;
  Tensor a, b, bias;
  double scale = 0;
};

void check_member(Member& m, int64_t K, const char* what) {
  check_weight(m.w, K, what);
  m.a = bf16(m.a, what);
  m.b = bf16(m.b, what);
  TORCH_CHECK_VALUE(m.a.dim() == 2 && m.b.dim() == 2 && m.a.size(1) == K && m.b.size(0) == m.w.N && m.b.size(1) == m.a.size(0), what,
                    ": lora_a ", m.a.sizes(), " / lora_b ", m.b.sizes(), " do not fit a [", m.w.N, ", ", K, "] layer");
  if (m.bias.defined()) {
    m.bias = bf16(m.bias, what);
    TORCH_CHECK_VALUE(m.bias.numel() == m.w.N, what, ": bias must have ", m.w.N, " elements");
  }
}

void fill(ttamd_lora_group_member& e, const Member& m, const Tensor& y) {
  e = {};
  e.quantized_data = (const uint8_t*)m.w.q.data_ptr();
  e.block_scalers = m.w.scal.data_ptr();
  e.block_scalers_t = opt_ptr(m.w.scal_t);
  e.quantized_data_t = (const uint8_t*)opt_ptr(m.w.q_t);
  e.lora_a = m.a.data_ptr();
  e.lora_b = m.b.data_ptr();
  e.bias = opt_ptr(m.bias);
  e.y = y.data_ptr();
  e.N = m.w.N;
  e.rank = (int)m.a.size(0);
  e.scale = (float)m.scale;
}

// The call for a handful of tokens, where it serves these members: its rule and the launch in one crossing of the ABI.  What it
// refuses, the calls for any number of tokens serve or name the fault of.
bool few_forward(const Tensor& x2, const ttamd_lora_group_member* members, int n, const Tensor& h_cat, const Tensor& act) {
  const int status = ttamd_lora_few_fwd_bf16(x2.data_ptr(), members, n, opt_ptr(h_cat), opt_ptr(act), x2.size(0), x2.size(1), stream_of(x2));
  if (status == TTAMD_EUNSUPPORTED || status == TTAMD_EINVAL) return false;
  check(status, "lora_few_fwd");
  return true;
}

struct LinearOut {
  Tensor x2, h, y;
};

// keep: the hidden activation is wanted for a backward; otherwise it lives at the head of the workspace
LinearOut linear_forward(const Tensor& x, Member m, bool keep) {
  const int64_t K = x.size(-1);
  LinearOut o;
  o.x2 = bf16(x, "qlora_linear_fwd").view({-1, K});
  check_member(m, K, "qlora_linear_fwd");
  const c10::DeviceGuard guard(x.device());
  const int64_t M = o.x2.size(0);
  const int rank = (int)m.a.size(0);
  o.y = at::empty(with_last(x, m.w.N), o.x2.options());
  if (keep) o.h = at::empty({M, rank}, o.x2.options());
  if (M <= TTAMD_FEW_TOKENS) {
    ttamd_lora_group_member one;
    fill(one, m, o.y);
    if (few_forward(o.x2, &one, 1, o.h, Tensor())) return o;
  }
  const size_t h_bytes = keep ? 0 : align256(M * rank * 2);
  const Tensor ws = scratch(h_bytes + ttamd_qlora_linear_fwd_workspace_bytes(M, m.w.N, K, rank), o.x2);
  char* w = (char*)ws.data_ptr();
  check(ttamd_qlora_linear_fwd_bf16(o.x2.data_ptr(), (const uint8_t*)m.w.q.data_ptr(), m.w.scal.data_ptr(), opt_ptr(m.w.scal_t), m.a.data_ptr(),
                                    m.b.data_ptr(), rank, (float)m.scale, opt_ptr(m.bias), o.y.data_ptr(), keep ? o.h.data_ptr() : w, M,
                                    m.w.N, K, w + h_bytes, ws.numel() - h_bytes, stream_of(x)),
        "qlora_linear_fwd");
  return o;
}

c10::IValue pack_weight(const Weight& w) { return c10::IValue(std::vector<Tensor>{w.q, w.scal, w.q_t, w.scal_t}); }
Weight unpack_weight(const c10::List<Tensor>& l, int64_t at, int64_t N) {
  Weight w;
  w.q = l.get(4 * at);
  w.scal = l.get(4 * at + 1);
  w.q_t = l.get(4 * at + 2);
  w.scal_t = l.get(4 * at + 3);
  w.N = N;
  return w;
}

// asking: the weight where it asks for a gradient.  It gets none, but the output then belongs to the graph.
struct QLoRALinearFn : torch::autograd::Function<QLoRALinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& a, const Tensor& b, const std::optional<Tensor>& bias,
                        const std::optional<Tensor>& /*asking*/, const Weight& w, double scale) {
    Member m;
    m.w = w;
    m.a = a;
    m.b = b;
    if (bias) m.bias = *bias;
    m.scale = scale;
    LinearOut o = linear_forward(x, m, true);
    ctx->save_for_backward({o.x2, o.h, a, b, w.whole});
    ctx->saved_data["w"] = pack_weight(w);
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["shape"] = x.sizes().vec();
    ctx->saved_data["bias"] = bias.has_value();
    return o.y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x2 = saved[0], &h = saved[1];
    const Tensor a = saved[2].contiguous(), b = saved[3].contiguous();
    const int64_t M = x2.size(0), K = x2.size(1), N = b.size(0);
    const int rank = (int)b.size(1);
    const Weight w = unpack_weight(ctx->saved_data["w"].toTensorList(), 0, N);
    const bool has_bias = ctx->saved_data["bias"].toBool();
    const bool need_x = ctx->needs_input_grad(0), need_ab = ctx->needs_input_grad(1) || ctx->needs_input_grad(2);
    const c10::DeviceGuard guard(x2.device());
    const Tensor gy = bf16(g[0], "qlora_linear_bwd").view({M, N});
    Tensor gx, ga, gb, gbias;
    if (need_x || need_ab) {
      if (need_x) gx = at::empty(ctx->saved_data["shape"].toIntVector(), x2.options());
      ga = at::empty_like(a);
      gb = at::empty_like(b);
      const Tensor ws = scratch(ttamd_qlora_linear_bwd_workspace_bytes(M, N, K, rank), x2);
      check(ttamd_qlora_linear_bwd_bf16(gy.data_ptr(), x2.data_ptr(), h.data_ptr(), (const uint8_t*)w.q.data_ptr(), w.scal.data_ptr(),
                                        (const uint8_t*)opt_ptr(w.q_t), opt_ptr(w.scal_t), nullptr, a.data_ptr(), b.data_ptr(), rank,
                                        (float)ctx->saved_data["scale"].toDouble(), opt_ptr(gx), ga.data_ptr(), gb.data_ptr(), M, N, K,
                                        ws.data_ptr(), ws.numel(), stream_of(x2)),
            "qlora_linear_bwd");
    }
    if (has_bias && ctx->needs_input_grad(3)) gbias = gy.sum(0);
    return {gx, ga, gb, gbias, Tensor(), Tensor(), Tensor()};
  }
};

bool asks_for_gradient(const Tensor& weight) { return at::GradMode::is_enabled() && weight.requires_grad(); }

Tensor qlora_linear(const Tensor& x, const Tensor& weight, const Tensor& q, const Tensor& scal, const std::optional<Tensor>& q_t, const std::optional<Tensor>& scal_t,
                    int64_t N, const Tensor& a, const Tensor& b, double scale, const std::optional<Tensor>& bias) {
  Member m;
  m.w.whole = weight;
  m.w.q = q;
  m.w.scal = scal;
  if (q_t) m.w.q_t = *q_t;
  if (scal_t) m.w.scal_t = *scal_t;
  m.w.N = N;
  if (bias) m.bias = *bias;
  const std::optional<Tensor> asking = asks_for_gradient(weight) ? std::optional<Tensor>(weight) : std::nullopt;
  if (asking || wants_grad({&x, &a, &b, &m.bias})) return QLoRALinearFn::apply(x, a, b, bias, asking, m.w, scale);
  m.a = a;
  m.b = b;
  m.scale = scale;
  return linear_forward(x, m, false).y;
}

// ---------------------------------------------------------------------------------------------------
// Groups of such linears with a common input
// ---------------------------------------------------------------------------------------------------
struct GroupOut {
  Tensor x2, h_cat, act;
  std::vector<Tensor> ys;
};

GroupOut group_forward(const Tensor& x, std::vector<Member>& ms, bool gated, bool keep) {
  const int n = (int)ms.size();
  TORCH_CHECK_VALUE(n >= 1 && n <= TTAMD_GROUP_MAX, "lora_group_fwd: a group has 1 to ", TTAMD_GROUP_MAX, " members, got ", n);
  TORCH_CHECK_VALUE(!gated || (n == 2 && ms[0].w.N == ms[1].w.N),
                    "lora_group_fwd: swiglu takes the gate and the up projection, two members of equal width");
  const int64_t K = x.size(-1);
  GroupOut o;
  o.x2 = bf16(x, "lora_group_fwd").view({-1, K});
  const c10::DeviceGuard guard(x.device());
  const int64_t M = o.x2.size(0);
  ttamd_lora_group_member arr[TTAMD_GROUP_MAX];
  int64_t r_total = 0;
  for (int i = 0; i < n; ++i) {
    check_member(ms[i], K, "lora_group_fwd");
    o.ys.push_back(at::empty(with_last(x, ms[i].w.N), o.x2.options()));
    fill(arr[i], ms[i], o.ys[i]);
    r_total += ms[i].a.size(0);
  }
  if (keep) o.h_cat = at::empty({M, r_total}, o.x2.options());
  if (gated) o.act = at::empty_like(o.ys[0]);
  if (M <= TTAMD_FEW_TOKENS && few_forward(o.x2, arr, n, o.h_cat, o.act)) return o;
  const size_t h_bytes = keep ? 0 : align256(M * r_total * 2);
  const size_t hidden = ttamd_lora_group_hidden_workspace_bytes(arr, n, M, K), fwd = ttamd_lora_group_fwd_workspace_bytes(arr, n, M, K);
  const size_t bytes = hidden > fwd ? hidden : fwd;
  const Tensor mem = scratch(h_bytes + bytes, o.x2);
  void* const h_cat = keep ? o.h_cat.data_ptr() : mem.data_ptr();
  void* const ws = (char*)mem.data_ptr() + h_bytes;
  void* s = stream_of(x);
  check(ttamd_lora_group_hidden_bf16(o.x2.data_ptr(), arr, n, h_cat, M, K, ws, bytes, s), "lora_group_hidden");
  if (gated) {
    check(ttamd_nf4_lora_group_swiglu_fwd_bf16(o.x2.data_ptr(), arr, n, h_cat, o.act.data_ptr(), M, K, ws, bytes, s),
          "lora_group_fwd");
  } else {
    check(ttamd_nf4_lora_group_fwd_bf16(o.x2.data_ptr(), arr, n, h_cat, M, K, ws, bytes, s), "lora_group_fwd");
  }
  return o;
}

struct GroupSpec {
  std::vector<Member> ms;
  bool gated = false;
  bool fused_swiglu_bwd = true;  // gated: the gradients of gate and up come out of the adapters' backward, not of a launch before it
};

// Differentiable inputs: x, then per member lora_a, lora_b and, where there is one, the bias; behind them the weights that ask
// for a gradient (as for a single layer).
struct QLoRAGroupFn : torch::autograd::Function<QLoRAGroupFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, at::TensorList inputs, GroupSpec& spec) {
    ctx->saved_data["inputs"] = (int64_t)inputs.size();
    GroupOut o = group_forward(x, spec.ms, spec.gated, true);
    variable_list save = {o.x2, o.h_cat};
    std::vector<Tensor> weights;
    std::vector<int64_t> n_out, bias;
    std::vector<double> scales;
    for (const Member& m : spec.ms) {
      save.push_back(m.a);
      save.push_back(m.b);
      for (const Tensor& t : {m.w.q, m.w.scal, m.w.q_t, m.w.scal_t}) weights.push_back(t);
      n_out.push_back(m.w.N);
      bias.push_back(m.bias.defined() ? 1 : 0);
      scales.push_back(m.scale);
    }
    if (spec.gated) {
      save.push_back(o.ys[0]);
      save.push_back(o.ys[1]);
    }
    for (const Member& m : spec.ms) save.push_back(m.w.whole);
    ctx->save_for_backward(std::move(save));
    ctx->saved_data["w"] = weights;
    ctx->saved_data["N"] = n_out;
    ctx->saved_data["bias"] = bias;
    ctx->saved_data["scales"] = scales;
    ctx->saved_data["gated"] = spec.gated;
    ctx->saved_data["fused_swiglu_bwd"] = spec.fused_swiglu_bwd;
    ctx->saved_data["shape"] = x.sizes().vec();
    if (spec.gated) return {o.act};
    return o.ys;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x2 = saved[0], &h_cat = saved[1];
    const std::vector<int64_t> n_out = ctx->saved_data["N"].toIntVector(), bias = ctx->saved_data["bias"].toIntVector();
    const std::vector<double> scales = ctx->saved_data["scales"].toDoubleVector();
    const bool gated = ctx->saved_data["gated"].toBool();
    const c10::List<Tensor> weights = ctx->saved_data["w"].toTensorList();
    const int n = (int)n_out.size();
    const int64_t M = x2.size(0), K = x2.size(1);
    const c10::DeviceGuard guard(x2.device());
    void* s = stream_of(x2);
    const bool need_x = ctx->needs_input_grad(0);
    std::vector<Member> ms(n);
    std::vector<Tensor> gys(n), ga(n), gb(n);
    ttamd_lora_group_member arr[TTAMD_GROUP_MAX];
    bool any_bias = false;
    for (int i = 0; i < n; ++i) any_bias = any_bias || bias[i];
    const bool fused_swiglu = gated && !any_bias && ctx->saved_data["fused_swiglu_bwd"].toBool();
    if (gated && !fused_swiglu) {
      auto [gg, gu] = swiglu_backward(g[0], saved[2 + 2 * n], saved[3 + 2 * n]);
      gys = {gg, gu};
    }
    for (int i = 0; i < n; ++i) {
      Member& m = ms[i];
      m.w = unpack_weight(weights, i, n_out[i]);
      m.a = saved[2 + 2 * i].contiguous();
      m.b = saved[3 + 2 * i].contiguous();
      m.scale = scales[i];
      if (fused_swiglu)
        gys[i] = at::empty({M, n_out[i]}, x2.options());
      else if (!gated)
        gys[i] = bf16(g[i], "lora_group_bwd");
      ga[i] = at::empty_like(m.a);
      gb[i] = at::empty_like(m.b);
      fill(arr[i], m, gys[i]);
      arr[i].grad_lora_a = ga[i].data_ptr();
      arr[i].grad_lora_b = gb[i].data_ptr();
    }
    const Tensor gh_cat = at::empty_like(h_cat);
    const Tensor ws = scratch(ttamd_lora_group_bwd_workspace_bytes(arr, n, M, K), x2);
    if (fused_swiglu) {
      const Tensor gact = bf16(g[0], "lora_group_bwd");
      check(ttamd_lora_group_swiglu_bwd_bf16(x2.data_ptr(), h_cat.data_ptr(), arr, n, gact.data_ptr(), saved[2 + 2 * n].data_ptr(),
                                             saved[3 + 2 * n].data_ptr(), gh_cat.data_ptr(), M, K, ws.data_ptr(), ws.numel(), s),
            "lora_group_bwd");
    } else {
      check(ttamd_lora_group_bwd_bf16(x2.data_ptr(), h_cat.data_ptr(), arr, n, gh_cat.data_ptr(), M, K, ws.data_ptr(), ws.numel(), s),
            "lora_group_bwd");
    }
    variable_list out;
    if (need_x) {
      Tensor gx = at::empty(ctx->saved_data["shape"].toIntVector(), x2.options());
      const size_t bytes = ttamd_nf4_group_bwd_dx_workspace_bytes(arr, n, M, K);
      const Tensor dx_ws = bytes ? scratch(bytes, x2) : Tensor();
      check(ttamd_nf4_group_bwd_dx_ws_bf16(arr, n, gh_cat.data_ptr(), gx.data_ptr(), M, K, opt_ptr(dx_ws), bytes, s), "nf4_group_bwd_dx");
      out.push_back(gx);
    } else {
      out.emplace_back();
    }
    size_t at_input = 1;
    for (int i = 0; i < n; ++i) {
      out.push_back(ga[i]);
      out.push_back(gb[i]);
      at_input += 2;
      if (bias[i]) {
        out.push_back(ctx->needs_input_grad(at_input) ? gys[i].reshape({-1, n_out[i]}).sum(0) : Tensor());
        ++at_input;
      }
    }
    out.resize(1 + ctx->saved_data["inputs"].toInt());  // the weights that ask
    out.emplace_back();                                 // the specification
    return out;
  }
};

// members: (weight, q, scal, q_t | None, scal_t | None, N, lora_a, lora_b, scale, bias | None) each
using MemberTuple = std::tuple<Tensor, Tensor, Tensor, std::optional<Tensor>, std::optional<Tensor>, int64_t, Tensor, Tensor, double, std::optional<Tensor>>;

std::vector<Tensor> lora_group(const Tensor& x, const std::vector<MemberTuple>& members, bool gated, bool fused_swiglu_bwd) {
  GroupSpec spec;
  spec.gated = gated;
  spec.fused_swiglu_bwd = fused_swiglu_bwd;
  std::vector<Tensor> inputs;
  bool grad = wants_grad({&x});
  for (const auto& t : members) {
    Member m;
    m.w.whole = std::get<0>(t);
    m.w.q = std::get<1>(t);
    m.w.scal = std::get<2>(t);
    if (std::get<3>(t)) m.w.q_t = *std::get<3>(t);
    if (std::get<4>(t)) m.w.scal_t = *std::get<4>(t);
    m.w.N = std::get<5>(t);
    m.a = std::get<6>(t);
    m.b = std::get<7>(t);
    m.scale = std::get<8>(t);
    if (std::get<9>(t)) m.bias = *std::get<9>(t);
    grad = grad || asks_for_gradient(m.w.whole) || wants_grad({&m.a, &m.b, &m.bias});
    inputs.push_back(m.a);
    inputs.push_back(m.b);
    if (m.bias.defined()) inputs.push_back(m.bias);
    spec.ms.push_back(std::move(m));
  }
  for (const Member& m : spec.ms)
    if (asks_for_gradient(m.w.whole)) inputs.push_back(m.w.whole);
  if (grad) return QLoRAGroupFn::apply(x, at::TensorList(inputs), spec);
  GroupOut o = group_forward(x, spec.ms, gated, false);
  if (gated) return {o.act};
  return o.ys;
}

// ---------------------------------------------------------------------------------------------------
// Fake quantisation and the converted integer linears
// ---------------------------------------------------------------------------------------------------
int dtype_code(at::ScalarType t, const char* what) {
  TORCH_CHECK_TYPE(t == at::kBFloat16 || t == at::kFloat, what, ": dtype ", t, " is not supported (bfloat16 and float32 are)");
  return t == at::kBFloat16 ? TTAMD_BF16 : TTAMD_F32;
}

// x [M, K] (..., K) bf16 with int8-held int4 weights; the activation is fake-quantised per token on the way
Tensor int8_dynamic_linear(const Tensor& x, const Tensor& q, const Tensor& scale, const Tensor& zeros, int64_t group_size,
                           const std::optional<Tensor>& bias) {
  const int64_t N = q.size(0), K = q.size(1);
  const Tensor x2 = aligned(bf16(x, "int8_group_linear").view({-1, K}));
  const int64_t M = x2.size(0);
  const int code = dtype_code(scale.scalar_type(), "int8_group_linear: scale");
  TORCH_CHECK_VALUE(q.scalar_type() == at::kChar && q.is_contiguous() && q.device() == x.device() && scale.is_contiguous() &&
                        scale.device() == x.device() && zeros.device() == x.device() && zeros.is_contiguous() && scale.numel() * group_size == N * K && zeros.numel() == scale.numel() &&
                        zeros.scalar_type() == scale.scalar_type(),
                    "int8_group_linear: q must be int8, scale and zeros of one dtype, all on x's device, with N * K / group_size elements");
  const Tensor b = bias ? aligned(bf16(*bias, "int8_group_linear")) : Tensor();
  TORCH_CHECK_VALUE(!b.defined() || (b.numel() == N && b.device() == x.device()), "int8_group_linear: bias must have ", N, " elements on x's device");
  const Tensor qa = aligned(q), sa = aligned(scale), za = aligned(zeros);
  const c10::DeviceGuard guard(x.device());
  Tensor y = at::empty(with_last(x, N), x2.options());
  const size_t bytes = ttamd_int8_dynamic_linear_workspace_bytes(M, N, K);
  const Tensor ws = bytes ? scratch(bytes, x2) : Tensor();
  check(ttamd_int8_dynamic_linear_bf16(x2.data_ptr(), (const int8_t*)qa.data_ptr(), sa.data_ptr(), za.data_ptr(), code, (int)group_size,
                                       opt_ptr(b), y.data_ptr(), M, N, K, opt_ptr(ws), bytes, stream_of(x)),
        "int8_dynamic_linear");
  return y;
}

Tensor uint4_group_linear(const Tensor& x, const Tensor& q, const Tensor& sz, int64_t group_size, const std::optional<Tensor>& bias) {
  const int64_t N = q.size(0), K = q.size(1) * 2;
  const Tensor x2 = aligned(bf16(x, "uint4_group_linear").view({-1, K}));
  const int64_t M = x2.size(0);
  TORCH_CHECK_VALUE(q.scalar_type() == at::kByte && q.is_contiguous() && q.device() == x.device() && sz.scalar_type() == at::kBFloat16 &&
                        sz.is_contiguous() && sz.device() == x.device() && sz.dim() == 3 && sz.size(0) * group_size == K && sz.size(1) == N && sz.size(2) == 2,
                    "uint4_group_linear: q must be uint8 and scales_and_zeros [K / group_size, N, 2] bf16, both on x's device");
  const Tensor b = bias ? aligned(bf16(*bias, "uint4_group_linear")) : Tensor();
  TORCH_CHECK_VALUE(!b.defined() || (b.numel() == N && b.device() == x.device()), "uint4_group_linear: bias must have ", N, " elements on x's device");
  const Tensor qa = aligned(q), sa = aligned(sz);
  const c10::DeviceGuard guard(x.device());
  Tensor y = at::empty(with_last(x, N), x2.options());
  const size_t bytes = ttamd_int4_linear_workspace_bytes(M, N, K);
  const Tensor ws = bytes ? scratch(bytes, x2) : Tensor();
  check(ttamd_uint4_group_linear_bf16(x2.data_ptr(), (const uint8_t*)qa.data_ptr(), sa.data_ptr(), (int)group_size, opt_ptr(b), y.data_ptr(),
                                      M, N, K, opt_ptr(ws), bytes, stream_of(x)),
        "uint4_group_linear");
  return y;
}

// ---------------------------------------------------------------------------------------------------
// Fake quantisation and the linear over fake-quantised operands
// ---------------------------------------------------------------------------------------------------
// 11 - 14 us of interpreter time per fake quantisation and 31 us per vendor product (most of it the choice of a kernel)
// made a training pass of few tokens host bound: a decoder layer of the 1B shape at 1000 tokens 1380 us for 850 us of kernels.
constexpr double kFqEps = 1.0 / 8388608;  // finfo(float32).eps

using MaybeTensor = std::optional<Tensor>;

// x [..., K] -> (fq(x), scale fp32 [rows], zero point int32 [rows])
std::tuple<Tensor, MaybeTensor, MaybeTensor> fq_per_token(const Tensor& x, bool want_qparams, bool bf16_qparams, std::optional<double> eps) {
  need_gpu(x, "fq_per_token_int8_asym");
  const int code = dtype_code(x.scalar_type(), "fq_per_token_int8_asym");
  const Tensor xc = x.detach().contiguous();
  const int64_t K = last_dim(xc, "fq_per_token_int8_asym"), rows = xc.numel() / K;
  const c10::DeviceGuard guard(x.device());
  Tensor out = at::empty_like(xc);
  MaybeTensor scale, zp;
  if (want_qparams) {
    scale = at::empty({rows}, xc.options().dtype(at::kFloat));
    zp = at::empty({rows}, xc.options().dtype(at::kInt));
  }
  const ttamd_fq_conventions conv = {(float)eps.value_or(kFqEps), (float)kFqEps, 1e-6f, 0};
  check(ttamd_fq_per_token_int8_asym_conv(xc.data_ptr(), code, rows, K, bf16_qparams ? TTAMD_BF16 : TTAMD_F32, out.data_ptr(),
                                          scale ? scale->data_ptr<float>() : nullptr, zp ? zp->data_ptr<int32_t>() : nullptr, &conv, stream_of(x)),
        "fq_per_token_int8_asym");
  return {out, scale, zp};
}

// w [..., K] -> (fq(w), scale fp32 [rows, K / group_size])
std::pair<Tensor, MaybeTensor> fq_per_group(const Tensor& w, int64_t group_size, bool want_scale, bool bf16_qparams, std::optional<double> eps) {
  need_gpu(w, "fq_per_group_int4_sym");
  const int code = dtype_code(w.scalar_type(), "fq_per_group_int4_sym");
  const Tensor wc = w.detach().contiguous();
  const int64_t K = last_dim(wc, "fq_per_group_int4_sym"), rows = wc.numel() / K;
  const c10::DeviceGuard guard(w.device());
  Tensor out = at::empty_like(wc);
  MaybeTensor scale;
  if (want_scale) scale = at::empty({rows, K / std::max<int64_t>(group_size, 1)}, wc.options().dtype(at::kFloat));
  const ttamd_fq_conventions conv = {(float)kFqEps, (float)eps.value_or(kFqEps), 1e-6f, 0};
  check(ttamd_fq_per_group_int4_sym_conv(wc.data_ptr(), code, rows, K, (int)group_size, bf16_qparams ? TTAMD_BF16 : TTAMD_F32, out.data_ptr(),
                                         scale ? scale->data_ptr<float>() : nullptr, &conv, stream_of(w)),
        "fq_per_group_int4_sym");
  return {out, scale};
}

// value = fq(x), gradient that of x
struct StraightThroughFn : torch::autograd::Function<StraightThroughFn> {
  static Tensor forward(AutogradContext*, const Tensor&, const Tensor& value) { return value; }
  static variable_list backward(AutogradContext*, variable_list g) { return {g[0], Tensor()}; }
};

Tensor straight_through(const Tensor& x, const Tensor& value) {
  const Tensor v = value.view(x.sizes());
  return wants_grad({&x}) ? StraightThroughFn::apply(x, v) : v;
}

// c = a . b^T (+ bias), a . b or a^T . b (kinds 0, 1, 2 of ttamd_gemm_mid_bf16) of contiguous matrices
Tensor gemm_mid(int kind, const Tensor& a_in, const Tensor& b_in, const Tensor& bias_in) {
  const Tensor a = aligned(a_in), b = aligned(b_in), bias = aligned(bias_in);
  const int64_t M = kind == 2 ? a.size(1) : a.size(0), K = kind == 2 ? a.size(0) : a.size(1), N = kind == 0 ? b.size(0) : b.size(1);
  TORCH_CHECK_VALUE((kind == 0 ? b.size(1) : b.size(0)) == K, "gemm_mid: ", a.sizes(), " and ", b.sizes(), " do not fit");
  const c10::DeviceGuard guard(a.device());
  Tensor c = at::empty({M, N}, a.options());
  int rows = 0, slices = 1, chain = 0;  // the workspace query counts slices that no launch of this kind may make
  if (M > 0 && N > 0 && K > 0) check(ttamd_gemm_mid_plan(kind, bias.defined(), M, N, K, &rows, &slices, &chain), "gemm_mid");
  const size_t bytes = slices > 1 ? (size_t)slices * M * N * sizeof(float) : 0;
  const Tensor ws = bytes ? scratch(bytes, a) : Tensor();
  check(ttamd_gemm_mid_bf16(kind, a.data_ptr(), b.data_ptr(), opt_ptr(bias), c.data_ptr(), M, N, K, opt_ptr(ws), bytes, stream_of(a)), "gemm_mid");
  return c;
}

Tensor ste_linear_forward(const Tensor& x, const Tensor& wq, const MaybeTensor& bias) {
  const Tensor x2 = bf16(x, "straight_through_linear").view({-1, x.size(-1)});
  const Tensor b = bias ? bf16(*bias, "straight_through_linear") : Tensor();
  TORCH_CHECK_VALUE(!b.defined() || (b.numel() == wq.size(0) && b.device() == x.device()), "straight_through_linear: bias must have ", wq.size(0),
                    " elements on x's device");
  return gemm_mid(0, x2, wq, b).view(with_last(x, wq.size(0)));
}

// F.linear(x, wq, bias) with the gradient of wq handed to weight
struct StraightThroughLinearFn : torch::autograd::Function<StraightThroughLinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const Tensor& wq, const MaybeTensor& bias) {
    // as F.linear does: each operand for the other's gradient only.  The weight itself (a leaf) is no operand: it may be
    // stepped before the backward, and serves a second differentiation alone.
    ctx->save_for_backward({weight.requires_grad() ? x : Tensor(), x.requires_grad() ? wq : Tensor()});
    ctx->saved_data["weight"] = weight;
    ctx->saved_data["shape"] = x.sizes().vec();
    ctx->saved_data["bias"] = bias.has_value();
    return ste_linear_forward(x, wq, bias);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto saved = ctx->get_saved_variables();
    const Tensor& x = saved[0];
    const std::vector<int64_t> shape = ctx->saved_data["shape"].toIntVector();
    const bool need_b = ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(3);
    Tensor wq = saved[1], gx, gw, gb;
    if (at::GradMode::is_enabled()) {  // a second differentiation: products that autograd can follow
      const Tensor gy = g[0].reshape({-1, g[0].size(-1)});
      if (ctx->needs_input_grad(0)) {
        const Tensor weight = ctx->saved_data["weight"].toTensor();
        gx = gy.matmul(wq + (weight - weight.detach())).view(shape);
      }
      if (ctx->needs_input_grad(1)) gw = gy.t().matmul(x.reshape({-1, shape.back()}));
      if (need_b) gb = gy.sum(0);
      return {gx, gw, Tensor(), gb};
    }
    const Tensor gy = bf16(g[0], "straight_through_linear_bwd").view({-1, g[0].size(-1)});
    if (ctx->needs_input_grad(0)) gx = gemm_mid(1, gy, wq, Tensor()).view(shape);
    if (ctx->needs_input_grad(1)) gw = gemm_mid(2, gy, x.contiguous().view({-1, shape.back()}), Tensor());
    if (need_b) gb = gy.sum(0);
    return {gx, gw, Tensor(), gb};
  }
};

Tensor straight_through_linear(const Tensor& x, const Tensor& weight, const Tensor& wq, const MaybeTensor& bias) {
  need_gpu(x, "straight_through_linear");
  const Tensor w = bf16(wq, "straight_through_linear: weight");
  TORCH_CHECK_VALUE(w.dim() == 2 && w.sizes() == weight.sizes() && w.device() == x.device(), "straight_through_linear: the weight's values are ",
                    w.sizes(), " on ", w.device().str());
  return wants_grad({&x, &weight}) || (bias && wants_grad({&*bias})) ? StraightThroughLinearFn::apply(x, weight, w, bias)
                                                                    : ste_linear_forward(x, w, bias);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  // like torch's own ops the calls run without the interpreter's lock: a launch waits where the queue is full
  const py::call_guard<py::gil_scoped_release> unlocked;
  m.def("ordinary", &ordinary);
  m.def("rms_norm", &rms_norm, unlocked);
  m.def("add_rms_norm", &add_rms_norm, unlocked);
  m.def("qkv_rope_repeat", &qkv_rope_repeat, unlocked);
  m.def("swiglu", &swiglu, unlocked);
  m.def("qlora_linear", &qlora_linear, unlocked);
  m.def("lora_group", &lora_group, unlocked);
  m.def("int8_dynamic_linear", &int8_dynamic_linear, unlocked);
  m.def("uint4_group_linear", &uint4_group_linear, unlocked);
  m.def("fq_per_token", &fq_per_token, unlocked);
  m.def("fq_per_group", &fq_per_group, unlocked);
  m.def("straight_through", &straight_through, unlocked);
  m.def("straight_through_linear", &straight_through_linear, unlocked);
}
