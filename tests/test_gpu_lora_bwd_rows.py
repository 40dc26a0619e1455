"""The adapter gradients gA = gh^T . x and gB = scale . gy^T . h of up to 2048 rows come from one launch without row splits, of more rows
from splits and a sum: rows at the edges of a wave's 32, of the sixteen waves' 512 and of the two ways; ranks at the edges of the
groups of 16; one linear and groups.

Outputs are one bf16 rounding (2^-9 relative, bounded by 2^-8) of fp32 sums of bf16 products; the sums' own error, a few 1e-7 of the
terms' absolute sum, is covered by 2e-5 of the largest output."""
import pytest
import torch

from torchtune_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def _close(got, want):
    torch.testing.assert_close(got.double(), want, rtol=2 ** -8, atol=2e-5 * want.abs().max().item())


@pytest.mark.parametrize("M", [1, 31, 32, 33, 511, 512, 513, 1025, 2048, 2049])
@pytest.mark.parametrize("N,K,r", [(64, 64, 8), (192, 64, 16), (64, 320, 24), (320, 1088, 40), (128, 192, 48), (192, 256, 64)])
def test_one_linear(M, N, K, r):
    g = torch.Generator(device=DEV).manual_seed(M + N + K + r)
    x, gy, h = (torch.randn(M, c, device=DEV, generator=g).to(BF) for c in (K, N, r))
    B = torch.randn(N, r, device=DEV, generator=g).to(BF)
    gh, ga, gb = ops.lora_bwd(gy, x, h, B, 0.5)
    _close(gh, 0.5 * (gy.double() @ B.double()))
    _close(ga, gh.double().t() @ x.double())
    _close(gb, 0.5 * (gy.double().t() @ h.double()))
    again = ops.lora_bwd(gy, x, h, B, 0.5)
    assert all(torch.equal(a, b) for a, b in zip((gh, ga, gb), again))


@pytest.mark.parametrize("M,Ns,ranks", [(40, (128, 64, 64), (16, 8, 24)), (700, (320, 192), (8, 32)), (1024, (64, 64, 128, 64), (16, 16, 16, 16)),
                                        (1025, (64, 64, 128, 64), (16, 16, 16, 16)), (2048, (128, 64), (24, 24))])
def test_groups(M, Ns, ranks):
    K = 192
    g = torch.Generator(device=DEV).manual_seed(M)
    members = []
    for n, r in zip(Ns, ranks):
        q = torch.randint(0, 256, (n * K // 2,), device=DEV, generator=g, dtype=torch.uint8)
        s = torch.rand(n * K // 64, device=DEV, generator=g).mul_(0.1)
        A, B = (torch.randn(c, device=DEV, generator=g).to(BF) for c in ((r, K), (n, r)))
        members.append(ops.GroupMember(q, s, ops.nf4_transpose_for_backward(q, s, n, K), A, B, None, 2.0 / r, n))
    x = torch.randn(M, K, device=DEV, generator=g).to(BF)
    h_cat = torch.randn(M, sum(ranks), device=DEV, generator=g).to(BF)
    gys = [torch.randn(M, n, device=DEV, generator=g).to(BF) for n in Ns]
    _, grads, gh = ops.lora_group_bwd(x, h_cat, members, gys, want_gx=False)
    off = 0
    for m, gy, r, (ga, gb) in zip(members, gys, ranks, grads):
        _close(ga, gh[:, off:off + r].double().t() @ x.double())
        _close(gb, m.scale * (gy.double().t() @ h_cat[:, off:off + r].double()))
        off += r


@pytest.mark.parametrize("M,r", [(2048, 8), (2048, 24), (2048, 48), (1024, 64), (2048, 64)])
def test_sums_of_32_rows_are_rounded_apart_from_the_others(M, r):
    """Rows 512 apart are the same wave's: beside 2^24, whose neighbours are 2 apart, each 32 of them (0.3125, 10 together, every
    partial sum of them exact) are added at once, not a few at a time.  A row of -2^24 then leaves their sum, which is off by at most half a
    spacing for each addition at that size."""
    steps = M // 512 - 1
    column = torch.zeros(M, device=DEV)
    column[0], column[32] = 2.0 ** 24, -(2.0 ** 24)
    for s in range(steps):
        column[512 * (s + 1):512 * (s + 1) + 32] = 0.3125
    big = column[:, None].expand(M, 64).to(BF).contiguous()
    ones = torch.ones(M, r, device=DEV, dtype=BF)
    B = torch.zeros(64, r, device=DEV, dtype=BF)
    B[0] = 1.0
    one_hot = torch.nn.functional.one_hot(torch.zeros(M, dtype=torch.long, device=DEV), 64).to(BF)
    _, _, gb = ops.lora_bwd(big, one_hot, ones, B, 1.0)
    gh, ga, _ = ops.lora_bwd(one_hot, big, ones, B, 1.0)
    assert torch.equal(gh, ones)
    assert bool(((gb.double() - 10.0 * steps).abs() <= steps).all()) and bool(((ga.double() - 10.0 * steps).abs() <= steps).all())
