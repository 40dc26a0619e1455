"""Fake-quantised linears below the sizes of the 256 x 256-tile kernels: the three products of ``ttamd_gemm_mid_bf16`` through
``FakeQuantizedLinear``, against fp32 matmuls of the same fake-quantised operands."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from torchtune_amd import _host, _lib, ops
from torchtune_amd.qat import FakeQuantizeConfig, FakeQuantizedLinear, FakeQuantizer

pytestmark = pytest.mark.gpu


def _close(got, want, length):
    # fp32 sums of exact products in some order (length * 2^-24 of the sum of magnitudes; random signs: its root), one bf16 rounding
    slack = 2.0 ** -8 * want.abs() + length ** 0.5 * 2.0 ** -23 * want.abs().max()
    assert bool(((got.double() - want).abs() <= slack).all())


# the weight gradient in slices of the tokens, which end in a part-filled step or not (tokens % 32)
SLICED_TOKENS = [(1000, 256, 1024, False), (1001, 256, 64, True), (1024, 320, 256, False), (2015, 256, 1536, False), (4097, 256, 128, True)]


# one k step and fewer (tokens are the contraction of the weight gradient), tile edges, widths of half a tile, split contractions
@pytest.mark.parametrize("M,N,K,bias", [(1, 256, 64, True), (31, 320, 128, False), (33, 256, 320, True), (128, 256, 256, False),
                                        (129, 448, 4096, True), (257, 4096, 192, False), (1000, 512, 2048, False), (700, 2048, 1088, True),
                                        (3000, 1024, 512, False)] + SLICED_TOKENS)
def test_linear_and_gradients(M, N, K, bias):
    if (M, N, K, bias) in SLICED_TOKENS:
        assert _lib.load().ttamd_gemm_mid_workspace_bytes(N, K, M) > 0
    torch.manual_seed(M + N + K)
    layer = FakeQuantizedLinear(K, N, bias, FakeQuantizeConfig(torch.int8, "per_token", is_symmetric=False),
                                FakeQuantizeConfig(torch.int4, group_size=32), device="cuda", dtype=torch.bfloat16)
    x = torch.randn(1, M, K, device="cuda").bfloat16().requires_grad_()
    gy = torch.randn(1, M, N, device="cuda").bfloat16()
    assert layer._mid_ok(x)
    y = layer(x)
    y.backward(gy)
    xq = ops.fq_per_token_int8_asym(x.detach())[0].double().view(M, K)
    wq, scale = ops.fq_per_group_int4_sym(layer.weight.detach(), 32)
    assert torch.equal(layer.weight_fake_quantizer.scale, scale)
    wq, g2 = wq.double(), gy.double().view(M, N)
    _close(y.view(M, N), xq @ wq.t() + (layer.bias.double() if bias else 0), K)
    _close(x.grad.view(M, K), g2 @ wq, N)
    _close(layer.weight.grad, g2.t() @ xq, M)
    if bias:
        assert torch.equal(layer.bias.grad, gy.view(M, N).sum(0))
    with torch.no_grad():
        assert torch.equal(layer(x), y)


@pytest.mark.parametrize("M,N,K,mid", [(2047, 2048, 4096, True), (4096, 2048, 2048, False), (3584, 2048, 2048, True), (16384, 1024, 1024, True),
                                       (16385, 1024, 1024, False)])
def test_rows_and_products_the_kernels_serve(M, N, K, mid):
    layer = FakeQuantizedLinear(K, N, False, None, FakeQuantizeConfig(torch.int4, group_size=32), device="cuda", dtype=torch.bfloat16)
    assert layer._mid_ok(torch.empty(M, K, device="cuda", dtype=torch.bfloat16)) is mid


def test_second_derivative():
    torch.manual_seed(0)
    layer = FakeQuantizedLinear(128, 256, False, None, FakeQuantizeConfig(torch.int4, group_size=32), device="cuda", dtype=torch.bfloat16)
    x = torch.randn(16, 128, device="cuda").bfloat16().requires_grad_()
    assert layer._mid_ok(x)
    gx, = torch.autograd.grad(layer(x).square().sum(), x, create_graph=True)
    gx.float().square().sum().backward()
    wq = ops.fq_per_group_int4_sym(layer.weight.detach(), 32)[0].float().requires_grad_()
    xr = x.detach().float().requires_grad_()
    gr, = torch.autograd.grad(F.linear(xr, wq).square().sum(), xr, create_graph=True)
    gr.square().sum().backward()
    # bf16 intermediates: a few roundings of 2^-8 each
    for got, want in ((x.grad, xr.grad), (layer.weight.grad, wq.grad)):
        assert float((got.float() - want).norm() / want.norm()) < 4 * 2.0 ** -8


@pytest.mark.parametrize("how", ["hook", "pre_hook", "subclass", "replacement", "patched", "global"])
def test_a_weight_quantizer_that_does_more_is_called(how):
    layer = FakeQuantizedLinear(128, 256, False, None, FakeQuantizeConfig(torch.int4, group_size=32), device="cuda", dtype=torch.bfloat16)
    x = torch.randn(16, 128, device="cuda").bfloat16()
    assert layer._mid_ok(x)
    want = F.linear(x, 2 * layer.weight_fake_quantizer(layer.weight))
    q, handle = layer.weight_fake_quantizer, None

    class Doubled(FakeQuantizer):
        def forward(self, w):
            return 2 * super().forward(w)

    class Other(torch.nn.Module):
        enabled, config = True, q.config

        def forward(self, w):
            return 2 * q(w)

    if how == "hook":
        q.register_forward_hook(lambda mod, args, out: 2 * out)
    elif how == "pre_hook":
        q.register_forward_pre_hook(lambda mod, args: (2 * args[0],))
    elif how == "subclass":
        layer.weight_fake_quantizer = Doubled(q.config)
    elif how == "replacement":
        layer.weight_fake_quantizer = Other()
    elif how == "patched":
        plain = q.forward
        q.forward = lambda w: 2 * plain(w)
    else:
        handle = torch.nn.modules.module.register_module_forward_hook(lambda mod, args, out: 2 * out if mod is q else None)
    try:
        # doubling is exact: in the weight, or in the quantised weight
        assert torch.equal(layer(x), want)
    finally:
        if handle is not None:
            handle.remove()


# tiles of 64, 128 and 256 rows with a last row tile of one row and a last column tile of half its width, fewer steps than the
# ring has stages and more, slices of unequal length (at kind 1 two of them are the four-wave kernel's; test_every_launch asserts
# which launch a product gets)
@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (65, 320, 192), (1025, 3520, 2048), (1025, 6464, 192), (1025, 6464, 1024), (129, 512, 4160),
                                   (1000, 2048, 8256), (2049, 2560, 128)])
@pytest.mark.parametrize("kind", [0, 1])
def test_tile_heights(kind, M, N, K):
    lib = _lib.load()
    torch.manual_seed(M + N + K + kind)
    a = torch.randn(M, K, device="cuda").bfloat16()
    b = torch.randn((N, K) if kind == 0 else (K, N), device="cuda").bfloat16()
    bias = torch.randn(N, device="cuda").bfloat16() if kind == 0 else None
    c = torch.full((M + 1, N), 7.0, device="cuda").bfloat16()  # one row beyond the product
    need = lib.ttamd_gemm_mid_workspace_bytes(M, N, K)
    ws = torch.empty(max(need, 1), device="cuda", dtype=torch.uint8)
    status = lib.ttamd_gemm_mid_bf16(kind, a.data_ptr(), b.data_ptr(), bias.data_ptr() if kind == 0 else None, c.data_ptr(), M, N, K,
                                     ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    assert status == 0
    want = a.double() @ (b.double().t() if kind == 0 else b.double())
    _close(c[:M], want + bias.double() if kind == 0 else want, K)
    assert bool((c[M] == 7).all())


# weight gradients on tiles of 256 x 256 whose last row and column of tiles hold 64 of 256: tokens of one part-filled step,
# around one step, an odd number of steps, more than the ring has stages (widths that are whole tiles: test_every_launch)
@pytest.mark.parametrize("tokens", [1, 31, 32, 33, 97, 1001, 1024])
def test_weight_gradients_on_wide_tiles(tokens):
    lib = _lib.load()
    N, K = 4160, 2624
    assert lib.ttamd_gemm_mid_workspace_bytes(N, K, tokens) == 0
    torch.manual_seed(tokens)
    gy = torch.randn(tokens, N, device="cuda").bfloat16()
    x = torch.randn(tokens, K, device="cuda").bfloat16()
    c = torch.full((N + 1, K), 7.0, device="cuda").bfloat16()  # one row beyond the product
    assert lib.ttamd_gemm_mid_bf16(2, gy.data_ptr(), x.data_ptr(), None, c.data_ptr(), N, K, tokens, None, 0,
                                   torch.cuda.current_stream().cuda_stream) == 0
    _close(c[:N], gy.double().t() @ x.double(), tokens)
    assert bool((c[N] == 7).all())


def _plan(kind, M, N, K, bias=0):
    tile_rows, slices, chain = (ctypes.c_int() for _ in range(3))
    assert _lib.load().ttamd_gemm_mid_plan(kind, bias, M, N, K, ctypes.byref(tile_rows), ctypes.byref(slices), ctypes.byref(chain)) == 0
    return tile_rows.value, slices.value, chain.value


def test_products_below_2048_rows():
    for M, N, K, mid in [(1000, 14336, 4096, True), (2047, 14336, 4096, True), (1000, 4096, 14336, False), (2047, 15360, 4096, False),
                         (1290, 6912, 2560, False), (2000, 800064, 64, False)]:
        layer = FakeQuantizedLinear(K, N, False, None, FakeQuantizeConfig(torch.int4, group_size=32), device="cuda", dtype=torch.bfloat16)
        assert layer._mid_ok(torch.empty(M, K, device="cuda", dtype=torch.bfloat16)) is mid, (M, N, K)
    test_linear_and_gradients(701, 9728, 3584, False)


@pytest.mark.parametrize("kind,M,N,K,rows", [(1, 368, 2048, 2048, 64), (0, 1053, 1024, 2816, 64), (0, 660, 3584, 9728, 128), (1, 1254, 2048, 8192, 128)])
def test_chains_that_end_before_the_contraction_does(kind, M, N, K, rows):
    """Every operand is 1 but one of 2^40 at the head of a chain and one of -2^40 at the head of the next: each absorbs the ones
    that follow it in its chain.  In one chain the second would restore the first, and half as many would be lost."""
    tile_rows, slices, chain = _plan(kind, M, N, K)
    assert (tile_rows, slices) == (rows, 1) and chain < K // 2
    a = torch.ones(M, K, device="cuda", dtype=torch.bfloat16)
    a[:, 0], a[:, 2 * chain] = 2.0 ** 40, -(2.0 ** 40)  # a step is 64 indices, the first 32 of them in this half's chains
    b = torch.ones((N, K) if kind == 0 else (K, N), device="cuda", dtype=torch.bfloat16)
    c = torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    assert _lib.load().ttamd_gemm_mid_bf16(kind, a.data_ptr(), b.data_ptr(), None, c.data_ptr(), M, N, K, None, 0,
                                           torch.cuda.current_stream().cuda_stream) == 0
    lost = K - c.float()
    last = min(chain, K // 2 - chain)  # of the second chain
    assert bool((lost <= chain + last + K / 128).all()) and bool((lost >= chain + last - 64 - K / 128).all())  # 128: a bf16 step
    torch.manual_seed(M + N + K)
    a, b = torch.randn(M, K, device="cuda").bfloat16(), torch.randn_like(b.float()).bfloat16()
    assert _lib.load().ttamd_gemm_mid_bf16(kind, a.data_ptr(), b.data_ptr(), None, c.data_ptr(), M, N, K, None, 0,
                                           torch.cuda.current_stream().cuda_stream) == 0
    _close(c, a.double() @ (b.double().t() if kind == 0 else b.double()), K)


# every launch that the plan can choose, by the plan's own word: (kind, M, N, K) -> rows of a tile, split / whole / ended chains
@pytest.mark.parametrize("kind,M,N,K,rows,form", [
    (0, 65, 320, 192, 64, "whole"), (0, 129, 512, 4160, 64, "split"), (0, 193, 320, 704, 64, "ended"), (0, 1025, 3520, 2048, 128, "whole"),
    (0, 1000, 2048, 8256, 128, "split"), (0, 193, 8256, 4160, 128, "ended"), (0, 1025, 6464, 192, 256, "whole"),
    (1, 65, 320, 192, 64, "whole"), (1, 129, 512, 4160, 64, "split"), (1, 193, 320, 704, 64, "ended"), (1, 1025, 3520, 2048, 128, "whole"),
    (1, 1000, 2048, 8256, 128, "split"), (1, 193, 8256, 4160, 128, "ended"), (1, 1025, 6464, 1024, 256, "whole"), (1, 1025, 6464, 192, 0, "whole"),
    (2, 64, 64, 513, 0, "split"), (2, 128, 576, 65, 0, "whole"), (2, 4160, 2624, 33, 256, "whole"), (2, 8192, 2048, 1001, 256, "whole"),
    (2, 8192, 2048, 1024, 256, "whole")])
def test_every_launch(kind, M, N, K, rows, form):
    tile_rows, slices, chain = _plan(kind, M, N, K)
    halves = 2 if kind < 2 and tile_rows else 1
    assert (tile_rows, "split" if slices > 1 else "ended" if halves * chain < K else "whole") == (rows, form)
    torch.manual_seed(M + N + K + kind)
    a = torch.randn((K, M) if kind == 2 else (M, K), device="cuda").bfloat16()
    b = torch.randn((N, K) if kind == 0 else (K, N), device="cuda").bfloat16()
    c = torch.full((M + 1, N), 7.0, device="cuda").bfloat16()  # one row beyond the product
    ws = torch.empty(max(4 * slices * M * N if slices > 1 else 0, 1), device="cuda", dtype=torch.uint8)
    assert _lib.load().ttamd_gemm_mid_bf16(kind, a.data_ptr(), b.data_ptr(), None, c.data_ptr(), M, N, K, ws.data_ptr(), ws.numel(),
                                           torch.cuda.current_stream().cuda_stream) == 0
    _close(c[:M], (a.double().t() if kind == 2 else a.double()) @ (b.double().t() if kind == 0 else b.double()), K)
    assert bool((c[M] == 7).all())


def test_a_linear_allocates_no_slabs_that_its_products_do_not_write():
    """1400 tokens of 2048 -> 8192: the four-wave kernel would cut the grad-input into four slices of 11 MB; it runs whole."""
    M, N, K = 1400, 8192, 2048
    assert _plan(1, M, K, N)[1] == 1 and _lib.load().ttamd_gemm_mid_workspace_bytes(M, K, N) == 4 * 4 * M * K
    w = torch.randn(N, K, device="cuda").mul_(0.02).bfloat16()
    x, gy = torch.randn(M, K, device="cuda").bfloat16().requires_grad_(), torch.randn(M, N, device="cuda").bfloat16()
    y = _host.load().straight_through_linear(x, w, w, None)
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    torch.autograd.grad(y, x, gy)
    assert torch.cuda.max_memory_allocated() - before < 2 * 2 * M * K  # the gradient itself: 2 bytes an element


def test_linears_whose_grad_input_part_fills_its_rounds_keep_the_dense_product():
    """Tiles of 128 rows in a second round of 280 of 512: slower here than with the vendor's kernels."""
    layer = FakeQuantizedLinear(3584, 9728, False, None, FakeQuantizeConfig(torch.int4, group_size=32), device="cuda", dtype=torch.bfloat16)
    for M, mid in [(740, True), (1182, False), (1447, False), (1485, True)]:
        assert layer._mid_ok(torch.empty(M, 3584, device="cuda", dtype=torch.bfloat16)) is mid, M
