"""Products of expert-sorted rows on 256 x 256 tiles (csrc/grouped_rowgemm.hip): a step of the reduction and half of one, tiles with few
rows, partial column tiles, and reductions of leftover tiles in parts.

Tolerance: one rounding to bf16 (2^-9 of the value, twice that allowed), and 1e-5 of the sum of the products' magnitudes for fp32 sums
of up to 8,224 products (2^-24 each, at random 100 times that)."""

import pytest
import torch

import neuronx_distributed_llama3_2_amd.ops as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,red,cols", [
    ([256, 1, 128, 129, 257, 0, 64], 32, 256),      # half a step alone
    ([130, 127, 5], 64, 264),                       # one step
    ([300, 17], 96, 8),                             # a step and a half
    ([512, 100, 384], 160, 520),
    ([2000, 48], 4096, 768),                        # fewer tiles than CUs, two parts
    ([40, 1100, 0, 300], 8224, 512),                # parts of which the last ends with half a step
    ([700, 900, 1000, 800, 1300, 1200, 1100, 1192], 4096, 2304)])   # whole rounds and a rest that is split
@pytest.mark.parametrize("mode", [0, 1])
def test_grouped_rows(mode, counts, red, cols):
    gen = torch.Generator(device="cuda").manual_seed(red + cols + mode)
    E, M = len(counts), sum(counts)
    offs = torch.tensor([0, *counts], device="cuda").cumsum(0).to(torch.int32)
    x = torch.randn(M, red, generator=gen, device="cuda").bfloat16()
    w = torch.randn((E, red, cols) if mode == 0 else (E, cols, red), generator=gen, device="cuda").bfloat16()
    C = ops.ext()
    outs = []
    for _ in range(2):   # (whichever part of a tile comes last, the order of the sums is the same)
        y = torch.full((M + 3, cols), 7.0, device="cuda", dtype=torch.bfloat16)
        C.grouped_gemm(mode, x, w, offs, y[:M], False)
        outs.append(y)
    assert torch.equal(outs[0], outs[1]) and (outs[0][M:] == 7.0).all()
    at = 0
    for e, n in enumerate(counts):
        xe, we = x[at:at + n].double(), (w[e] if mode == 0 else w[e].t()).double()
        want, size = xe @ we, xe.abs() @ we.abs()
        assert ((outs[0][at:at + n].double() - want).abs() <= 2 ** -8 * want.abs() + 1e-5 * size).all(), e
        at += n
