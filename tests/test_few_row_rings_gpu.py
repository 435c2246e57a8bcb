"""Tiles of at most 64 and at most 128 rows of the 256 x 256-tile products (run_few of csrc/gemm_tile.h): row counts around the 8-row pieces that the four waves load in turn,
reductions of one step to more than the ring's four, three places, whole and with half a step at the end, rows after the last one left alone.

Tolerance: bf16 results of fp32 sums are within 2^-9 each (3 x 2^-9 of the 2-norm: with the sums' own rounding)."""

import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops
from neuronx_distributed_llama3_2_amd.ops._ext import gemm_ext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[1, 7, 8, 9, 24, 25, 31, 32], [33, 40, 41, 56, 57, 63, 64], [65, 72, 73, 96, 97, 104], [105, 120, 121, 127, 128, 256 + 12]])
@pytest.mark.parametrize("red", [32, 64, 96, 128, 160, 192, 256, 288, 320, 448])
def test_few_rows(red, counts):
    gen = torch.Generator(device="cuda").manual_seed(red + sum(counts))
    E, rows, cols = len(counts), sum(counts), 280
    offs = torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).to(torch.int32).cuda()
    x = torch.randn(rows, red, generator=gen, device="cuda").bfloat16()
    for mode, shape in ((0, (E, red, cols)), (1, (E, cols, red))):
        w = torch.randn(shape, generator=gen, device="cuda").bfloat16()
        y = torch.full((rows + 1, cols), 7.0, device="cuda").bfloat16()
        ops.ext().grouped_gemm(mode, x, w, offs, y[:rows], False)
        want = torch.cat([x[offs[e]:offs[e + 1]].double() @ (w[e] if mode == 0 else w[e].t()).double() for e in range(E)])
        for e in range(E):
            a, b = int(offs[e]), int(offs[e + 1])
            assert float((y[a:b].double() - want[a:b]).norm()) < 3 * 2 ** -9 * float(want[a:b].norm())
        assert bool((y[rows] == 7).all())


@pytest.mark.parametrize("rows", [1, 9, 40, 64, 65, 100, 128])
def test_few_rows_with_an_activation(rows):
    gen = torch.Generator(device="cuda").manual_seed(rows)
    for red in (64, 160, 256, 320):
        x = torch.randn(rows, red, generator=gen, device="cuda").bfloat16()
        w = torch.randn(512, red, generator=gen, device="cuda").bfloat16()
        w = w / red ** 0.5
        for act in (0, 1):
            y = torch.full((rows + 1, 512 if act else 256), 7.0, device="cuda").bfloat16()
            gemm_ext().act_gemm(act, x, w, y[:rows])
            p = (x.double() @ w.double().t()).bfloat16().double()
            want = p.clamp_min(0).square() if act else torch.nn.functional.silu(p[:, :256]) * p[:, 256:]
            # (a product next to a rounding boundary may fall on its other side: 2^-8 of it, twice that of its square or of the other's product)
            assert float((y[:rows].double() - want).norm()) < 2 ** -7 * float(want.norm())
            assert bool((y[rows] == 7).all())
