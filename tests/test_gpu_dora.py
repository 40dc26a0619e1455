"""GPU parity of the fused QDoRA path (NF4 base weight) against the CPU oracle: weight norms, forward, all gradients."""
import pytest
import torch

from oracle import lora_oracle, nf4_oracle
from torchtune_amd import _lib, ops
from torchtune_amd.modules.peft import DoRALinear, get_adapter_params
from torchtune_amd.nf4_tensor import NF4Tensor, to_nf4

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def _layer(K, N, r, alpha, use_bias, seed):
    g = torch.Generator().manual_seed(seed)
    W = (torch.randn(N, K, generator=g) * 0.02).to(BF)
    A = (torch.randn(r, K, generator=g) * 0.05).to(BF)
    B = (torch.randn(N, r, generator=g) * 0.05).to(BF)
    b = (torch.randn(N, generator=g) * 0.1).to(BF) if use_bias else None
    prev = torch.get_default_dtype()
    torch.set_default_dtype(BF)
    try:
        with torch.device(DEV):
            layer = DoRALinear(K, N, rank=r, alpha=alpha, use_bias=use_bias, quantize_base=True)
    finally:
        torch.set_default_dtype(prev)
    with torch.no_grad():
        layer.weight.copy_(W.to(DEV))
        layer.lora_a.weight.copy_(A.to(DEV))
        layer.lora_b.weight.copy_(B.to(DEV))
        if use_bias:
            layer.bias.copy_(b.to(DEV))
    return layer, nf4_oracle.nf4_quantize(W, 64, 256), A, B, b


@pytest.mark.parametrize("K,N,r,use_bias", [(512, 512, 8, False), (2240, 320 * 8, 16, True), (4096, 1024, 64, False)])
def test_weight_norm_and_magnitude_init(K, N, r, use_bias):
    layer, parts, A, B, _ = _layer(K, N, r, 2.0 * r, use_bias, seed=0)
    assert isinstance(layer.weight, NF4Tensor)
    layer.initialize_dora_magnitude()
    want = lora_oracle.dora_weight_norm(parts, A, B, 2.0 * r, r)
    # both sides: bf16 merged rows, fp32 sum of squares, sqrt, one rounding to bf16; the summation order differs
    torch.testing.assert_close(layer.magnitude.detach().cpu().float(), want.float(), rtol=2 ** -7, atol=0)
    assert (layer.magnitude.detach().cpu() == want).float().mean() > 0.9


@pytest.mark.parametrize("K,N,r", [(64, 256, 8), (2048, 40, 24), (1216, 1024, 32), (1088, 2048, 40), (5120, 336, 16)])
def test_weight_norm_kernel_edges(K, N, r):
    """Half chunks, strips that end early, row tiles that are not full, ranks on both sides of one matrix step."""
    layer, parts, A, B, _ = _layer(K, N, r, 2.0 * r, False, seed=3)
    norm, _ = ops.nf4_dora_weight_norm(layer.weight.quantized_data, layer.weight.block_scalers(), N, K, layer.lora_a.weight.detach(),
                                       layer.lora_b.weight.detach(), 2.0)
    want = lora_oracle.dora_weight_norm(parts, A, B, 2.0 * r, r)
    torch.testing.assert_close(norm.cpu().float(), want.float(), rtol=2 ** -7, atol=0)
    assert (norm.cpu() == want).float().mean() > 0.9


@pytest.mark.parametrize("M,N", [(1, 72), (5, 520), (1031, 1032)])
def test_backward_prologue_edges(M, N):
    g = torch.Generator().manual_seed(M)
    gy, out = (torch.randn(M, N, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
    mns, mag = (torch.rand(N, generator=g).add(0.5).to(torch.bfloat16).to(DEV) for _ in range(2))
    gy0, gmag = ops.dora_bwd_prologue(gy, out, mns, mag)
    assert torch.equal(gy0, gy * mns)
    want = (gy.double() * out.double()).sum(0) / mag.double()
    size = (gy.double() * out.double()).abs().sum(0) / mag.double()
    # fp32 sums of M products, one rounding to bf16
    assert bool(((gmag.double() - want).abs() <= want.abs() * 2.0 ** -8 + size * M * 2.0 ** -23).all())


@pytest.mark.parametrize("M,K,N,r,use_bias", [(96, 512, 512, 8, True), (300, 1024, 768, 16, False), (1024, 2048, 2048, 16, True)])
def test_forward_backward_vs_oracle(M, K, N, r, use_bias):
    alpha = 2.0 * r
    layer, parts, A, B, b = _layer(K, N, r, alpha, use_bias, seed=1)
    g = torch.Generator().manual_seed(2)
    mag = (torch.rand(N, generator=g) * 0.3 + 0.05).to(BF)
    with torch.no_grad():
        layer.magnitude.copy_(mag.to(DEV))
    x = torch.randn(M, K, generator=g).to(BF)
    gy = (torch.randn(M, N, generator=g) * 0.1).to(BF)

    xo = x.clone().requires_grad_()
    Ao, Bo, mo = A.clone().requires_grad_(), B.clone().requires_grad_(), mag.clone().requires_grad_()
    yo = lora_oracle.dora_linear_forward(xo, parts, Ao, Bo, mo, alpha, r, bias=b)
    yo.backward(gy)

    xd = x.to(DEV).requires_grad_()
    y = layer(xd)
    y.backward(gy.to(DEV))
    # (1) against the closed form evaluated in fp32 from the same bf16 operands and the oracle's bf16 norm:
    #     rtol 1e-2 / atol 1e-2 (the kernel accumulates in fp32 and rounds the result once)
    D = nf4_oracle.nf4_dequantize(parts).float()
    c = (mag / lora_oracle.dora_weight_norm(parts, A, B, alpha, r)).float()
    y32 = (x.float() @ D.T + (b.float() if b is not None else 0.0) + (alpha / r) * (x.float() @ A.float().T) @ B.float().T) * c
    torch.testing.assert_close(y.detach().cpu().float(), y32, rtol=1e-2, atol=1e-2)
    # (2) against the eager oracle, which rounds each of its ~10 intermediate tensors to bf16: rtol 2e-2 / atol 3e-2
    torch.testing.assert_close(y.detach().cpu().float(), yo.detach().float(), rtol=2e-2, atol=3e-2)
    torch.testing.assert_close(xd.grad.cpu().float(), xo.grad.float(), rtol=2e-2, atol=2e-2)
    for got, want in ((layer.lora_a.weight.grad, Ao.grad), (layer.lora_b.weight.grad, Bo.grad), (layer.magnitude.grad, mo.grad)):
        want = want.float()
        torch.testing.assert_close(got.cpu().float(), want, rtol=3e-2, atol=3e-2 * float(want.abs().max()))
    assert layer.weight.grad is None
    assert set(get_adapter_params(layer)) == {"lora_a.weight", "lora_b.weight", "magnitude"}


def test_initial_magnitude_makes_dora_equal_lora_and_disabled_is_the_base_layer():
    layer, parts, A, B, _ = _layer(512, 512, 8, 16.0, False, seed=3)
    layer.initialize_dora_magnitude()
    x = torch.randn(64, 512).to(BF)
    y = layer(x.to(DEV)).cpu()
    want = lora_oracle.lora_linear_forward(x, parts, A, B, 16.0, 8)
    torch.testing.assert_close(y.float(), want.float(), rtol=2e-2, atol=2e-2)
    layer.disabled = True
    base = layer(x.to(DEV)).cpu()
    torch.testing.assert_close(base.float(), (x.float() @ nf4_oracle.nf4_dequantize(parts).float().T), rtol=1e-2, atol=1e-2)


def test_raw_c_abi_validation():
    lib = _lib.load()
    t = torch.zeros(64, device=DEV, dtype=BF)
    p = t.data_ptr()
    assert lib.ttamd_nf4_dora_weight_norm_bf16(p, p, p, p, 12, 1.0, None, p, None, 64, 64, p, 1 << 20, None) == -1
    assert b"rank" in lib.ttamd_last_error()
    assert lib.ttamd_nf4_dora_weight_norm_bf16(p, p, p, p, 8, 1.0, None, p, None, 64, 64, p, 4, None) == -3
    assert lib.ttamd_dora_bwd_prologue_bf16(p, p, p, p, p, p, 8, 12, p, 1 << 20, None) == -1
    assert lib.ttamd_nf4_dora_linear_fwd_bf16(p, p, p, None, None, None, 0, 0.0, None, None, p, 8, 64, 64, None) == -1
    assert b"col_scale" in lib.ttamd_last_error()


@pytest.mark.parametrize("with_hook", [False, True])
def test_merged_dora_checkpoint_reproduces_the_layer(with_hook):
    """get_merged_lora_ckpt with a magnitude entry (torchtune/modules/peft/_utils.py:245-263): the merged dense
    weight, used as a plain linear, gives the DoRA layer's output; the NF4 weight goes through the one-pass
    dequantise + merge kernel (`with_hook=False`) or arrives already dense on the CPU (`with_hook=True`)."""
    from torchtune_amd.modules.common_utils import reparametrize_as_dtype_state_dict_post_hook
    from torchtune_amd.modules.peft import get_merged_lora_ckpt

    K, N, r, alpha = 1024, 768, 16, 32.0
    layer, parts, A, B, _ = _layer(K, N, r, alpha, False, seed=5)
    layer.initialize_dora_magnitude()
    with torch.no_grad():
        layer.magnitude.mul_(torch.linspace(0.5, 1.5, N, device=DEV).to(BF))
    sd = {"l." + k: v.detach() for k, v in layer.state_dict().items()}
    if with_hook:
        reparametrize_as_dtype_state_dict_post_hook(layer, sd, dtype=BF, offload_to_cpu=True)
        assert sd["l.weight"].device.type == "cpu"
        sd = {k: v.cpu() for k, v in sd.items()}
    out = get_merged_lora_ckpt(sd, rank=r, alpha=alpha)
    assert out.keys() == {"l.weight"}
    merged = out["l.weight"]
    assert merged.dtype == BF and merged.shape == (N, K)
    # closed form in fp32 from the oracle's dequantised weight
    Wd = nf4_oracle.nf4_dequantize(parts).float()
    full = Wd + (alpha / r) * (B.float() @ A.float())
    want = full * (layer.magnitude.detach().float().cpu() / full.norm(dim=1)).view(-1, 1)
    torch.testing.assert_close(merged.float().cpu(), want, rtol=2e-2, atol=2e-3)
    x = (torch.randn(64, K, generator=torch.Generator().manual_seed(6))).to(BF).to(DEV)
    y_layer = layer(x)
    y_merged = torch.nn.functional.linear(x, merged.to(DEV))
    torch.testing.assert_close(y_merged.float(), y_layer.float(), rtol=2e-2, atol=3e-2)


# ---- the reference's own DoRALinear tests, restated (tests/torchtune/modules/peft/test_dora.py) ------------------------

class _default_dtype:
    def __init__(self, dtype):
        self.dtype = dtype

    def __enter__(self):
        self.prev = torch.get_default_dtype()
        torch.set_default_dtype(self.dtype)

    def __exit__(self, *a):
        torch.set_default_dtype(self.prev)


def _fixed_init(model):
    with torch.no_grad():
        for _, p in model.named_parameters():
            p.copy_(lora_oracle.fixed_init_tensor(p.shape, dtype=p.dtype).to(p.device))


def _dora(use_bias, dtype, quantize_base, in_dim=512, out_dim=512, **kw):
    with _default_dtype(dtype), torch.device(DEV):
        m = DoRALinear(in_dim, out_dim, rank=4, alpha=1.0, use_bias=use_bias, quantize_base=quantize_base, **kw)
    _fixed_init(m)
    return m


@pytest.mark.parametrize("use_bias", [True, False])
def test_dora_weight_nf4_when_quantized(use_bias):
    # test_dora.py:113-119
    m = _dora(use_bias, BF, True)
    assert isinstance(m.weight, NF4Tensor)
    if use_bias:
        assert not isinstance(m.bias, NF4Tensor) and m.bias.dtype == BF


def test_dora_weight_nf4_when_quantized_with_quantization_kwargs():
    # test_dora.py:121-130
    m = _dora(True, BF, True, block_size=8, scaler_block_size=4)
    assert isinstance(m.weight, NF4Tensor) and m.weight.block_size == 8 and m.weight.scaler_block_size == 4
    assert not isinstance(m.bias, NF4Tensor)


def test_dora_weight_nf4_when_quantized_raises_value_error_with_bad_args():
    # test_dora.py:132-147
    with pytest.raises(ValueError, match="``quantize_base`` is False, but received the following quantization arguments"):
        _dora(True, BF, False, block_size=8, scaler_block_size=4)


@pytest.mark.parametrize("use_bias,dtype", [(False, BF), (True, torch.float32), (False, torch.float32)])
def test_qdora_parity(use_bias, dtype):
    # test_dora.py:152-182: a dense DoRA layer holding the dequantised weight gives the same output
    torch.manual_seed(16)
    q = _dora(use_bias, dtype, True)
    d = _dora(use_bias, dtype, False)
    d.weight.data = q.weight.to(dtype)
    if use_bias:
        d.bias.data = q.bias.detach().clone()
    q.initialize_dora_magnitude()
    d.initialize_dora_magnitude()
    torch.testing.assert_close(q.magnitude, d.magnitude, rtol=1.6e-2, atol=1e-5)
    x = torch.randn(2, 32, 512, dtype=dtype, device=DEV)
    out_d, out_q = d(x), q(x)
    if dtype == BF:
        torch.testing.assert_close(out_d, out_q, rtol=1.6e-2, atol=1e-5)  # torch.testing's bf16 defaults, as in the reference
    else:
        torch.testing.assert_close(out_d, out_q, rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("dtype", [BF, torch.float32])
def test_dora_quantized_state_dict(dtype):
    # test_dora.py:184-237
    from functools import partial

    from torch import nn

    from torchtune_amd.modules.common_utils import reparametrize_as_dtype_state_dict_post_hook

    with _default_dtype(dtype), torch.device(DEV):
        layer = DoRALinear(512, 512, rank=4, alpha=1.0, use_bias=False, quantize_base=True)
    layer._register_state_dict_hook(partial(reparametrize_as_dtype_state_dict_post_hook, dtype=dtype, offload_to_cpu=False))
    sd = layer.state_dict()
    for v in sd.values():
        assert v.dtype == dtype and not isinstance(v, NF4Tensor)
    with _default_dtype(dtype), torch.device(DEV):
        reload = DoRALinear(512, 512, rank=4, alpha=1.0, use_bias=False, quantize_base=True)
    reload.weight = nn.Parameter(to_nf4(torch.zeros_like(layer.weight.get_original_weight(), dtype=dtype, device=layer.weight.device)))
    assert not torch.allclose(layer.weight.quantized_data, reload.weight.quantized_data)
    reload.load_state_dict(sd)
    assert torch.allclose(layer.weight.quantized_data, reload.weight.quantized_data)


def test_dora_single_device_init():
    # test_dora.py:239-261 on the device: dense fp32 layer, random adapters, magnitude = row norms of the merged weight
    from torch import nn

    torch.manual_seed(3)
    with _default_dtype(torch.float32), torch.device(DEV):
        layer = DoRALinear(64, 128, rank=4, alpha=1.0, use_bias=False)
    layer.lora_a.weight = nn.Parameter(torch.randn_like(layer.lora_a.weight))
    layer.lora_b.weight = nn.Parameter(torch.randn_like(layer.lora_b.weight))
    expected = torch.linalg.norm(layer.weight + layer.scaling * layer.lora_b.weight @ layer.lora_a.weight, dim=1)
    assert not torch.allclose(layer.magnitude, expected)
    layer.initialize_dora_magnitude()
    assert torch.allclose(layer.magnitude, expected)
