"""Products of few rows (csrc/few_rows.hip) where a workgroup's loads begin and end in other ways: tiles next to each other whose last
workgroup has fewer, tiles with fewer stages than are loaded ahead, waves without a chunk, single tiles of whole rounds of stages and
not, against 64-bit references.

Tolerance: as in test_few_rows_gpu, 3 x 2^-9 of the result's 2-norm (two bf16 roundings of at most 2^-9 each, fp32 sums)."""

import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu
TOL = 3 * 2 ** -9


def _run(M, N, K, epi, norm, int8, repeat=3):
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 5 * K)
    rows = 2 * N if epi == 2 else N
    if int8:
        w = torch.randint(-128, 128, (rows, K), generator=gen, device="cuda", dtype=torch.int8)
        s = torch.rand(rows, generator=gen, device="cuda") * 3e-4 + 1e-5
        exact = w.double() * s.double()[:, None]
    else:
        w, s = (torch.randn(rows, K, generator=gen, device="cuda") * 0.02).bfloat16(), None
        exact = w.double()
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    g = (1 + 0.1 * torch.randn(K, generator=gen, device="cuda")).bfloat16() if norm else None
    z = x.double()
    if norm:
        z = z * torch.rsqrt(z.square().mean(-1, keepdim=True) + 1e-5) * g.double()
    z = z @ exact.t()
    if epi == 2:
        z = torch.nn.functional.silu(z[:, :N]) * z[:, N:]
    first = None
    for _ in range(repeat):
        y = torch.full((M, N), float("nan"), device="cuda").bfloat16()
        ops.ext().dgemv(epi, x, g, 1e-5, w, y, 0, 0, 0, None, None, None, 1, None, None, None, wscale=s)
        assert torch.isfinite(y.float()).all()
        assert float((y.double() - z).norm() / z.norm()) < TOL
        first = y if first is None else first
        assert torch.equal(y, first)


# tiles of 16 rows: 257 and 258 are two rounds (the last workgroup has one tile, or two), 513 and 515 three; 128 and 136 elements: waves without a
# chunk, 8 and 15 chunks: one or two a wave; above 2,048 elements 11 waves of up to three chunks
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("N", [257 * 16, 258 * 16 - 5, 513 * 16 + 8, 515 * 16])
@pytest.mark.parametrize("M,K", [(3, 128), (16, 144), (4, 1024), (9, 1920), (5, 2048), (20, 2048), (8, 2176), (16, 4096), (30, 4224)])
def test_rounds_of_tiles(M, N, K, int8):
    _run(M, N, K, 0, False, int8)
    _run(M, N, K, 0, True, int8)


# one tile a workgroup, activations streamed: chunks a wave 1, 2, both, 3 and 4, 4, 5, 8, 8 and 9; 44 and 56 chunks: 11 and 7 waves
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("K", [1024, 2048, 1664, 3200, 4096, 5120, 8192, 8448, 5632, 7168])
@pytest.mark.parametrize("M,N", [(3, 2048), (8, 40), (4, 4096), (20, 1000), (18, 3072), (5, 8192)])
def test_single_tiles(M, N, K, int8):
    _run(M, N, K, 0, False, int8)
    if K <= 2048:
        _run(M, N, K, 0, True, int8)


# SwiGLU: 6 and 7 rounds (tiles of 8 columns), halves of the rows
@pytest.mark.parametrize("M,N,K", [(4, 6 * 2048, 256), (16, 6 * 2048 + 8, 512), (13, 7 * 2048, 384), (30, 7 * 1024 + 24, 2176), (30, 6 * 1024, 2176)])
def test_swiglu_rounds(M, N, K):
    _run(M, N, K, 2, True, False)


# 25 to 32 rows of reductions past 2,048 (few and many weight rows) go to this kernel, between them to the library: in the op, either side of each line
@pytest.mark.parametrize("M,N,K,few", [(25, 8, 2056, True), (32, 3072, 4224, True), (32, 3073, 3080, False), (32, 4096, 3072, True), (25, 4097, 3072, False),
                                       (24, 12288, 2056, True), (25, 12288, 3064, False), (32, 12288, 3072, True), (17, 12287, 4096, False), (32, 3072, 4232, False)])
def test_long_reductions_by_rows_of_weights(M, N, K, few):
    from neuronx_distributed_llama3_2_amd.ops.gemv import few_rows_pay, skinny_linear

    assert few_rows_pay(M, N, K) is few
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 5 * K)
    w, x = (torch.randn(N, K, generator=gen, device="cuda") * 0.02).bfloat16(), torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    z = x.double() @ w.double().t()
    assert float((skinny_linear(x, w).double() - z).norm() / z.norm()) < TOL


# reductions in parts: a wave with as many stages as are loaded ahead and with fewer, a last part with fewer chunks, parts without a chunk for every wave
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", [(13, 1024, 8192), (13, 2048, 8192), (16, 40, 4352), (15, 2048, 5632), (32, 1000, 11008), (9, 3072, 14336)])
def test_parts(M, N, K, int8):
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 5 * K)
    if int8:
        w = torch.randint(-128, 128, (N, K), generator=gen, device="cuda", dtype=torch.int8)
        s = torch.rand(N, generator=gen, device="cuda") * 3e-4 + 1e-5
        exact = w.double() * s.double()[:, None]
    else:
        w, s = (torch.randn(N, K, generator=gen, device="cuda") * 0.02).bfloat16(), None
        exact = w.double()
    x, y0 = (torch.randn(M, n, generator=gen, device="cuda").bfloat16() for n in (K, N))
    z = y0.double() + x.double() @ exact.t()
    tickets = torch.zeros(1024, dtype=torch.int32, device="cuda")
    for _ in range(3):
        y = y0.clone()
        ops.ext().dgemv(1, x, None, 0.0, w, y, 0, 0, 0, None, None, None, 1, None, None, None, wscale=s, tickets=tickets)
        assert float((y.double() - z).norm() / z.norm()) < TOL and not tickets.any()
