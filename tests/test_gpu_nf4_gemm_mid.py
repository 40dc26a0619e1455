"""The fused NF4 product on tiles of 64 x 128, 96 x 256 and 128 x 256 (nf4_gemm_mid.hip) at the edges of tiles, steps and slices:
forward with both layouts of the scalers, grad-input, groups either way.

Every output is one bf16 rounding (2^-9 relative, bounded by 2^-8) of fp32 sums of at most 9000 products on the bits of the
dequantised weight; the reference's own fp32 sums and these differ by a few 1e-7 of the terms' absolute sum, which the
absolute part (2e-5 of the largest output) covers.  The plan query says which kernel a size runs on, so that each is met."""
import ctypes

import pytest
import torch

from oracle import nf4_oracle
from torchtune_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def _plan(M, n_out, kc, by_128=True, may_slice=True, forward=True):
    rows, slices, chain = (ctypes.c_int() for _ in range(3))
    assert _lib.load().ttamd_nf4_gemm_plan(M, n_out, kc, may_slice, by_128, forward, ctypes.byref(rows), ctypes.byref(slices), ctypes.byref(chain)) == 0
    return rows.value, slices.value, chain.value


def _close(got, want):
    torch.testing.assert_close(got.float(), want, rtol=2 ** -8, atol=2e-5 * want.abs().max().item())


class _Weight:
    """Random codes and block scalers (a whole NF4 tensor has sizes of its own): ``dense`` is what they stand for."""

    def __init__(self, N, K, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)
        self.codes = torch.randint(0, 256, (N * K // 2,), device=DEV, generator=self.g, dtype=torch.uint8)
        self.scalers = (torch.rand(N * K // 64, device=DEV, generator=self.g) * 0.05 + 0.01).to(BF).float()
        self.transposed = ops.nf4_transpose_for_backward(self.codes, self.scalers, N, K)
        table = torch.tensor(nf4_oracle.NF4_TABLE, device=DEV).to(BF).float()
        values = torch.stack((table[(self.codes >> 4).long()], table[(self.codes & 15).long()]), dim=1).view(N * K // 64, 64)
        self.dense = (values * self.scalers[:, None]).to(BF).float().view(N, K)


# (tokens, outputs, contraction, tile rows, sliced): last rows and columns of a tile alone, contractions of one step, of an odd number of
# 64 (the 64-row tiles take 128 at a time), of fewer steps than the ring has stages, slices that end in a half step
SIZES = [
    (33, 64, 128, 64, False), (64, 128, 256, 64, False), (65, 192, 192, 64, False), (129, 320, 320, 64, False), (97, 64, 576, 64, False),
    (33, 64, 1088, 64, True), (63, 64, 2112, 64, True), (193, 1088, 4160, 64, True), (129, 4160, 2112, 64, False), (63, 8256, 2112, 64, False),
    (33, 64, 64, 96, False), (96, 576, 64, 96, False), (97, 320, 64, 96, False), (333, 14336, 128, 96, False),
    (700, 8256, 64, 128, False), (1500, 4160, 64, 128, False), (97, 4160, 4160, 128, True), (450, 4160, 8256, 96, True), (1100, 8256, 1088, 256, False),
]


@pytest.mark.parametrize("M,N,K,rows,sliced", SIZES)
@pytest.mark.parametrize("r", [8, 40])
def test_forward(M, N, K, rows, sliced, r):
    got = _plan(M, N, K)
    assert got[0] == rows and (got[1] > 1) == sliced, got
    t = _Weight(N, K, M + N + K)
    D, g = t.dense, t.g
    x = torch.randn(M, K, device=DEV, generator=g).to(BF)
    h = torch.randn(M, r, device=DEV, generator=g).to(BF)
    B = (torch.randn(N, r, device=DEV, generator=g) * 0.02).to(BF)
    bias = (torch.randn(N, device=DEV, generator=g) * 0.1).to(BF)
    cs = (torch.rand(N, device=DEV, generator=g) + 0.5).to(BF)
    want = x.float() @ D.t() + (h.float() * 0.5).to(BF).float() @ B.float().t()
    for scal_t in (None, t.transposed[1]):
        y = ops.nf4_lora_linear_fwd(x, t.codes, t.scalers, N, h, B, 0.5, block_scalers_t=scal_t)
        _close(y, want)
        y2 = ops.nf4_lora_linear_fwd(x, t.codes, t.scalers, N, h, B, 0.5, bias, block_scalers_t=scal_t, col_scale=cs)
        _close(y2, (want + bias.float()) * cs.float())
        assert torch.equal(y, ops.nf4_lora_linear_fwd(x, t.codes, t.scalers, N, h, B, 0.5, block_scalers_t=scal_t))


@pytest.mark.parametrize("M,K,N,rows,sliced", SIZES)
def test_grad_input(M, K, N, rows, sliced):
    got = _plan(M, K, N, forward=False)
    assert got[0] == rows and (got[1] > 1) == sliced, got
    t = _Weight(N, K, M + N + K)
    D, g = t.dense, t.g
    gy = torch.randn(M, N, device=DEV, generator=g).to(BF)
    gh = torch.randn(M, 24, device=DEV, generator=g).to(BF)
    A = (torch.randn(24, K, device=DEV, generator=g) * 0.02).to(BF)
    gx = ops.nf4_linear_bwd_dx(gy, t.codes, t.scalers, K, gh, A, transposed=t.transposed)
    _close(gx, gy.float() @ D + gh.float() @ A.float())
    _close(ops.nf4_linear_bwd_dx(gy, t.codes, t.scalers, K, transposed=t.transposed), gy.float() @ D)


@pytest.mark.parametrize("M,N,K", [(520, 13312, 8192)])
def test_without_a_workspace_the_plan_of_the_query_runs(M, N, K):
    """Slices would be the better way, but there is no memory for them: the tiles are those that the query names, and a row has the
    bits of the same tiles in a larger product.  Tiles of another kind add the contraction in other chains."""
    assert _plan(M, N, K)[1] > 1 and _plan(M, N, K, may_slice=False)[0] == 256 and _plan(700, N, K)[0] == 256
    t = _Weight(N, K, 1)
    x = torch.randn(700, K, device=DEV, generator=t.g).to(BF)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream

    def run(rows):
        y = torch.empty(rows, N, device=DEV, dtype=BF)
        assert lib.ttamd_nf4_lora_linear_fwd_ws_bf16(x.data_ptr(), t.codes.data_ptr(), t.scalers.data_ptr(), t.transposed[1].data_ptr(), None, None, 0, 0.0,
                                                     None, None, y.data_ptr(), rows, N, K, None, 0, stream) == 0
        return y

    assert torch.equal(run(M), run(700)[:M])
    sliced = ops.nf4_lora_linear_fwd(x[:M], t.codes, t.scalers, N, block_scalers_t=t.transposed[1])
    assert not torch.equal(sliced, run(M))
    _close(sliced, x[:M].float() @ t.dense.t())


@pytest.mark.parametrize("M,Ns,K", [(700, (3072, 3072), 3072), (333, (4096, 1024, 1024), 4096)])
def test_groups_without_a_workspace(M, Ns, K):
    """Members that slices would serve better, without memory for them: the bits of the members alone without a workspace."""
    members = []
    for i, n in enumerate(Ns):
        t = _Weight(n, K, 3 * M + i)
        A, B = ((torch.randn(s, device=DEV, generator=t.g) * 0.02).to(BF) for s in ((8, K), (n, 8)))
        members.append(ops.GroupMember(t.codes, t.scalers, t.transposed, A, B, None, 2.0, n))
    assert any(_plan(M, n, K)[1] > 1 for n in Ns)
    x = torch.randn(M, K, device=DEV, generator=t.g).to(BF)
    h = torch.randn(M, 8 * len(Ns), device=DEV, generator=t.g).to(BF)
    ys = [torch.empty(M, n, device=DEV, dtype=BF) for n in Ns]
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    array = (_lib.LoraGroupMember * len(Ns))()
    for e, m, y in zip(array, members, ys):
        e.quantized_data, e.block_scalers, e.block_scalers_t = m.qdata.data_ptr(), m.block_scalers.data_ptr(), m.transposed[1].data_ptr()
        e.lora_a, e.lora_b, e.y, e.N, e.rank, e.scale = m.lora_a.data_ptr(), m.lora_b.data_ptr(), y.data_ptr(), m.N, 8, m.scale
    assert lib.ttamd_nf4_lora_group_fwd_bf16(x.data_ptr(), array, len(Ns), h.data_ptr(), M, K, None, 0, stream) == 0
    for i, (m, y) in enumerate(zip(members, ys)):
        hi, alone = h[:, 8 * i:8 * i + 8].contiguous(), torch.empty_like(y)
        assert lib.ttamd_nf4_lora_linear_fwd_ws_bf16(x.data_ptr(), m.qdata.data_ptr(), m.block_scalers.data_ptr(), m.transposed[1].data_ptr(), hi.data_ptr(),
                                                     m.lora_b.data_ptr(), 8, m.scale, None, None, alone.data_ptr(), M, m.N, K, None, 0, stream) == 0
        assert torch.equal(y, alone)


@pytest.mark.parametrize("M,K,Ns", [(65, 192, (128, 64, 64)), (200, 1088, (1088, 128, 192)), (333, 4096, (4096, 1024, 1024)), (700, 64, (8256, 4160)),
                                    (129, 2112, (4160, 64)), (300, 576, (320, 320))])
@pytest.mark.parametrize("bias", [False, True])
def test_groups(M, K, Ns, bias):
    """Members with slices of their own, with and without ends of chains, and widths that are no multiple of 128 (the grad-input then
    takes its contraction 64 at a time).  The forward has the bits of the members alone."""
    ranks = (8, 16, 24)[: len(Ns)]
    members, D = [], []
    for i, (n, r) in enumerate(zip(Ns, ranks)):
        t = _Weight(n, K, 7 * M + n + i)
        d, g = t.dense, t.g
        A, B = ((torch.randn(s, device=DEV, generator=g) * 0.02).to(BF) for s in ((r, K), (n, r)))
        b = (torch.randn(n, device=DEV, generator=g) * 0.1).to(BF) if bias else None
        members.append(ops.GroupMember(t.codes, t.scalers, t.transposed, A, B, b, 32.0 / r, n))
        D.append(d)
    x = torch.randn(M, K, device=DEV, generator=g).to(BF)
    gys = [torch.randn(M, n, device=DEV, generator=g).to(BF) for n in Ns]
    h_cat, ys = ops.lora_group_fwd(x, members)
    gx, _, gh = ops.lora_group_bwd(x, h_cat, members, gys)
    want, off = 0, 0
    for m, d, y, gy, r in zip(members, D, ys, gys, ranks):
        h = h_cat[:, off:off + r].contiguous()
        _close(y, x.float() @ d.t() + (h.float() * m.scale).to(BF).float() @ m.lora_b.float().t() + (m.bias.float() if bias else 0.0))
        alone = ops.nf4_lora_linear_fwd(x, m.qdata, m.block_scalers, m.N, h, m.lora_b, m.scale, m.bias, block_scalers_t=m.transposed[1])
        assert torch.equal(y, alone)
        want = want + gy.float() @ d + gh[:, off:off + r].float() @ m.lora_a.float()
        off += r
    _close(gx, want)


def test_infinities_stay_in_their_rows_and_columns():
    """A contraction of an odd number of 64 on the 64-row tiles: the half step reads indices that the step before had, which must
    not count twice, nor turn an infinity elsewhere into a NaN."""
    M, N, K = 65, 192, 192
    t = _Weight(N, K, 3)
    D, g = t.dense, t.g
    x = torch.randn(M, K, device=DEV, generator=g).to(BF)
    x[5, 100] = float("inf")
    y = ops.nf4_lora_linear_fwd(x, t.codes, t.scalers, N, block_scalers_t=t.transposed[1])
    want = x.float() @ D.t()
    keep = torch.arange(M, device=DEV) != 5
    _close(y[keep], want[keep])
    assert torch.equal(torch.isnan(y[5]), torch.isnan(want[5])) and torch.equal(torch.isinf(y[5]), torch.isinf(want[5]))
