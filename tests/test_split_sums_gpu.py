"""Tiles of the grouped products whose reduction is split over workgroups (csrc/grouped_rowgemm.hip): two to eight parts, as many as not a power of two, of tiles of all heights, the
last workgroup adding them up row fragment by row fragment.  Several launches in turn share the sums' places and counters.

Tolerance: bf16 results of fp32 sums are within 2^-9 each (3 x 2^-9 of the 2-norm: with the sums' own rounding)."""

import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu


# reduction steps of 64: 64 give two parts at most, 96 three, 128 four, 160 five, 256 eight; 7 x 8 tiles of an expert leave fewer
@pytest.mark.parametrize("steps,cols", [(64, 264), (96, 264), (128, 520), (160, 264), (224, 136), (256, 264), (128, 7 * 256 + 8)])
@pytest.mark.parametrize("counts", [[256, 200], [129, 161, 100], [31, 32, 33, 64, 65, 97], [700, 5]])
def test_parts(steps, cols, counts):
    red = 64 * steps
    gen = torch.Generator(device="cuda").manual_seed(red + cols + sum(counts))
    E, rows = len(counts), sum(counts)
    offs = torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).to(torch.int32).cuda()
    x = torch.randn(rows, red, generator=gen, device="cuda").bfloat16()
    for mode, shape in ((0, (E, red, cols)), (1, (E, cols, red))):
        w = torch.randn(shape, generator=gen, device="cuda").bfloat16()
        want = torch.cat([x[offs[e]:offs[e + 1]].double() @ (w[e] if mode == 0 else w[e].t()).double() for e in range(E)])
        first = None
        for _ in range(3):
            y = torch.full((rows + 1, cols), 7.0, device="cuda").bfloat16()
            ops.ext().grouped_gemm(mode, x, w, offs, y[:rows], False)
            assert float((y[:rows].double() - want).norm()) < 3 * 2 ** -9 * float(want.norm())
            assert bool((y[rows] == 7).all())
            first = y if first is None else first
            assert torch.equal(y, first)   # (the parts' order is fixed)
