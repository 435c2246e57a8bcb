"""Hyper-connection steps at the widths and rows where their kernel changes.  Against float64."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("S", [1, 4, 8])
@pytest.mark.parametrize("M", [5, 64, 65])
@pytest.mark.parametrize("W", [4, 1020, 1024, 1028, 2044, 2048, 2052, 4092, 4096, 4100, 1026])
def test_hyper_step(W, M, S, dtype):
    g = torch.Generator().manual_seed(W * 8 + S)
    eps = 1e-5
    rnd = lambda *n: torch.randn(*n, generator=g)  # noqa: E731
    mix, wr, rd, nw, bias = rnd(S, S), rnd(S), rnd(S), 0.3 * rnd(W), rnd(W)
    y, embed = rnd(M, W + 4).to(dtype)[:, :W], rnd(7, W).to(dtype)
    ids = torch.tensor([3, 0, 7, -1, 6] * 13)[:M]              # 7, -1: outside of the table, zero rows
    cu = lambda t: t.cuda()  # noqa: E731
    tol = 1e-5 if dtype == torch.float32 else 2 ** -8           # of the results' rounding

    def norm(x, read):
        u = (x * read.double()[:, None]).sum(1)
        return u / (u.square().mean(1, keepdim=True) + eps).sqrt() * (1 + nw.double())

    def close(a, want, t):
        assert ((a.double().cpu() - want).abs() <= t * want.abs() + t * 1e-1 * want.abs().max()).all()

    table = torch.cat([embed.double(), torch.zeros(1, W, dtype=torch.float64)])
    x = table[torch.where((ids >= 0) & (ids < 7), ids, 7)][:, None].repeat(1, S, 1)
    streams = torch.full((M, S, W), float("nan"), device="cuda")
    h = ops.hyper_step(streams, read=cu(rd), norm_w=cu(nw), eps=eps, embed=cu(embed), ids=cu(ids))
    assert torch.equal(streams.double().cpu(), x)
    close(h, norm(x, rd), tol)
    h = ops.hyper_step(streams, y=cu(y), y_bias=cu(bias), mix=cu(mix), write=cu(wr), read=cu(rd), norm_w=cu(nw), eps=eps)
    x = torch.einsum("st,msw->mtw", mix.double(), x) + wr.double()[:, None] * (y.double() + bias.double())[:, None]
    close(streams, x, 1e-5)
    close(h, norm(x, rd), tol)
    rows, before = torch.tensor([4, 1]), streams.clone()
    h = ops.hyper_step(streams, y=cu(y), mix=cu(mix), write=cu(wr), read=cu(rd), norm_w=cu(nw), eps=eps, rows=cu(rows), store=False)
    x = torch.einsum("st,msw->mtw", mix.double(), streams.double().cpu()) + wr.double()[:, None] * y.double()[:, None]
    close(h, norm(x, rd)[rows], tol)
    assert torch.equal(streams, before)

