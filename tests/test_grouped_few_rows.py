"""Products of expert-sorted rows where there are few: the room that leftover tiles' parts take follows the rows, and so do the loads of the
rows; tiles of one row to half a tile and more, between rows of NaN.  Tolerance as in test_grouped_tiles_gpu."""
import pytest
import torch

import neuronx_distributed_llama3_2_amd.ops as ops


@pytest.mark.parametrize("red,ncols,rows,E,mb,tickets", [
    (4096, 1024, 0, 8, 0, 0), (4064, 1024, 64, 8, 8 * 8 * 2 / 32, 64), (4032, 1024, 64, 8, 0, 0),     # none; 64 steps, the last a half; 63
    (4096, 256, 1, 8, 8 * 2 / 32, 16), (4096, 1024, 2, 8, 8 * 2 / 32, 16), (4096, 1024, 16, 8, 8 * 8 / 32, 64), (4096, 1024, 33, 8, 8 * 8 * 2 / 32, 64),
    (4096, 28672, 16, 8, 8, 256), (14336, 4096, 128, 8, 32, 256), (4096, 28672, 8192, 8, 64, 256), (8192, 256, 256, 1, 8, 32)])
def test_room(red, ncols, rows, E, mb, tickets):
    size, n = ops.ext().grouped_gemm_workspace(red, ncols, rows, E)
    assert n == tickets and size == mb * 2 ** 20, size / 2 ** 20


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[1], [2, 0, 1], [33, 1, 64, 0, 5], [127, 128], [129, 8, 9, 65], [7] * 40, [300, 96, 1]])
@pytest.mark.parametrize("red,cols", [(4096, 264), (4128, 512), (6144, 8), (16384, 1032), (96, 520), (512, 2304)])
@pytest.mark.parametrize("mode", [0, 1])
def test_few_rows(mode, red, cols, counts):
    gen = torch.Generator(device="cuda").manual_seed(red + cols + sum(counts))
    E, M = len(counts), sum(counts)
    offs = torch.tensor([0, *counts], device="cuda").cumsum(0).to(torch.int32)
    x = torch.full((M + 130, red), float("nan"), device="cuda", dtype=torch.bfloat16)[:M]
    x.copy_(torch.randn(M, red, generator=gen, device="cuda"))
    w = torch.randn((E, red, cols) if mode == 0 else (E, cols, red), generator=gen, device="cuda").bfloat16()
    outs = []
    for _ in range(2):   # (whichever part of a tile comes last, the order of the sums is the same)
        y = torch.full((M + 3, cols), 7.0, device="cuda", dtype=torch.bfloat16)
        ops.ext().grouped_gemm(mode, x, w, offs, y[:M], False)
        outs.append(y)
    assert torch.equal(outs[0], outs[1]) and (outs[0][M:] == 7.0).all()
    at = 0
    for e, n in enumerate(counts):
        xe, we = x[at:at + n].double(), (w[e] if mode == 0 else w[e].t()).double()
        want, size = xe @ we, xe.abs() @ we.abs()
        assert ((outs[0][at:at + n].double() - want).abs() <= 2 ** -8 * want.abs() + 1e-5 * size).all(), e
        at += n
