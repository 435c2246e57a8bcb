"""The loops of the 256 x 256-tile products (csrc/gemm_tile.h) where their rings begin and end: reductions of one step to more than the
ring holds, with half a step at the end, tiles with so few rows that a quarter or half of the fragments are worked on, and token counts
with a partial first step, against 64-bit references.

Tolerance: bf16 outputs of fp32 sums are within 2^-9 of the result each (3 x 2^-9 of the 2-norm: with the sums' own rounding);
fp32 gradients: K products of relative error 2^-24 each, at random, 1e-6."""

import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu


def _offs(counts):
    return torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).to(torch.int32).cuda()


@pytest.mark.parametrize("red", [32, 64, 96, 128, 192, 224, 320, 544])
@pytest.mark.parametrize("counts", [[1, 64, 65, 0, 256 + 40], [33, 128, 129, 255], [257, 256 + 64, 17]])
def test_row_tiles(red, counts):
    gen = torch.Generator(device="cuda").manual_seed(red + sum(counts))
    E, rows, cols = len(counts), sum(counts), 264
    offs = _offs(counts)
    x = torch.randn(rows, red, generator=gen, device="cuda").bfloat16()
    for mode, shape in ((0, (E, red, cols)), (1, (E, cols, red))):
        w = torch.randn(shape, generator=gen, device="cuda").bfloat16()
        y = torch.full((rows, cols), float("nan"), device="cuda").bfloat16()
        ops.ext().grouped_gemm(mode, x, w, offs, y, False)
        for e in range(E):
            a, b = int(offs[e]), int(offs[e + 1])
            if a < b:
                want = x[a:b].double() @ (w[e].double() if mode == 0 else w[e].double().t())
                assert torch.isfinite(y[a:b].float()).all()
                assert float((y[a:b].double() - want).norm() / want.norm()) < 3 * 2 ** -9


@pytest.mark.parametrize("tokens", [1, 31, 32, 33, 64, 65, 96, 128, 129, 192, 200, 256, 320, 321, 1000])
def test_token_steps(tokens):
    """An output whose rows begin at odd places takes the loop whatever the number of tokens (with atomic adds)."""
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    M, N = 264, 520
    dy = torch.randn(tokens, M, generator=gen, device="cuda").bfloat16()
    x = torch.randn(tokens, N, generator=gen, device="cuda").bfloat16()
    for splits in (1, 2):
        c = torch.randn(M, N + 1, generator=gen, device="cuda")
        want = c.double()
        want[:, :N] += dy.double().t() @ x.double()
        ops.ext().wgrad_gemm(c[:, :N], dy, x, splits, True)
        assert float((c.double() - want).norm() / want.norm()) < 1e-6 and torch.equal(c[:, N], want[:, N].float())


def test_groups_of_tokens():
    gen = torch.Generator(device="cuda").manual_seed(5)
    counts = [1500, 0, 2789, 63, 1696]
    offs, rows = _offs(counts), sum(counts)
    dy = torch.randn(rows, 264, generator=gen, device="cuda").bfloat16()
    x = torch.randn(rows, 520, generator=gen, device="cuda").bfloat16()
    c = torch.zeros(len(counts), 264, 520, device="cuda")
    ops.ext().grouped_gemm(2, dy, x, offs, c, True)
    for e in range(len(counts)):
        a, b = int(offs[e]), int(offs[e + 1])
        want = dy[a:b].double().t() @ x[a:b].double()
        assert float((c[e].double() - want).norm()) <= 1e-6 * float(want.norm())
