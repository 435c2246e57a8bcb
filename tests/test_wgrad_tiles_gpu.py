"""The weight-gradient kernel's two loops at the token counts where one takes over from the other, with partial first and last
steps, partial tiles and strided operands between NaNs.  Against float64."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd.ops._ext import ext

pytestmark = pytest.mark.gpu


def _check(mg, before, dy, x):
    # sums of T products of bf16 in fp32: T roundings of 2^-24 of the sum of magnitudes, at the most
    ref = before.double() + dy.double().t() @ x.double()
    scale = dy.double().abs().t() @ x.double().abs() + before.double().abs()
    assert ((mg.double() - ref).abs() <= (dy.shape[0] + 1) * 2.0 ** -24 * scale + 1e-30).all()


def _among_nans(T, n, g):
    t = torch.full((T + 64, n + 8), float("nan"), device="cuda", dtype=torch.bfloat16)[:T, :n]
    return t.copy_(torch.randn(T, n, generator=g, device="cuda"))


@pytest.mark.parametrize("T", [449, 450, 451, 512, 700, 701, 767, 768, 769])
@pytest.mark.parametrize("M,N", [(8, 264), (520, 512), (3328, 3848)])   # 2, 6 and 208 tiles
def test_dense(T, M, N):
    g = torch.Generator(device="cuda").manual_seed(T + M)
    dy, x = _among_nans(T, M, g), _among_nans(T, N, g)
    mg = torch.randn(M, N, generator=g, device="cuda")
    before = mg.clone()
    ext().wgrad_gemm(mg, dy, x, 1, True)
    _check(mg, before, dy, x)


@pytest.mark.parametrize("sizes", [[0, 1, 63, 64, 6900], [1400] * 4, [1401] * 4, [0, 129, 5000, 0, 2000]])
@pytest.mark.parametrize("K,N", [(264, 72), (768, 3848)])
def test_grouped(sizes, K, N):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes) + K)
    rows = sum(sizes)
    x, dy = (torch.randn(rows, n, generator=g, device="cuda").bfloat16() for n in (K, N))
    offs = torch.tensor([0] + sizes, device="cuda").cumsum(0).to(torch.int32)
    mg = torch.randn(len(sizes), K, N, generator=g, device="cuda")
    before = mg.clone()
    ext().grouped_gemm(2, x, dy, offs, mg, True)
    for e in range(len(sizes)):
        a, b = int(offs[e]), int(offs[e + 1])
        _check(mg[e], before[e], x[a:b], dy[a:b]) if b > a else None
        assert b > a or torch.equal(mg[e], before[e])
