"""The weight-gradient kernel's epilogue (load, add and store where a workgroup alone owns its tile, atomics otherwise) and
its last, partial token stage.  Against float64, on partial tiles, strided and misaligned gradients, empty and one-row
experts, any token count; what lies beside the gradient stays."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd.ops._ext import ext

pytestmark = pytest.mark.gpu


def _check(mg, before, dy, x):
    # sums of T products of bf16 in fp32: T roundings of 2^-24 of the sum of magnitudes, at the most
    ref = before.double() + dy.double().t() @ x.double()
    scale = dy.double().abs().t() @ x.double().abs() + before.double().abs()
    assert ((mg.double() - ref).abs() <= (dy.shape[0] + 1) * 2.0 ** -24 * scale + 1e-30).all()


@pytest.mark.parametrize("pad,shift", [(0, 0), (4, 0), (8, 4), (1, 0), (0, 1)])   # the last two: atomics
@pytest.mark.parametrize("T,M,N,splits", [(32, 8, 8, 1), (64, 256, 256, 1), (96, 264, 248, 1), (160, 520, 72, 1), (512, 264, 264, 4)])
def test_dense(T, M, N, splits, pad, shift):
    g = torch.Generator(device="cuda").manual_seed(T + M)
    dy, x = (torch.randn(T, n, generator=g, device="cuda").bfloat16() for n in (M, N))
    flat = torch.randn(M * (N + pad) + shift + 64, generator=g, device="cuda")
    start = flat.clone()
    view = lambda f: f[shift:shift + M * (N + pad)].view(M, N + pad)[:, :N]
    ext().wgrad_gemm(view(flat), dy, x, splits)
    _check(view(flat), view(start), dy, x)
    view(flat).copy_(view(start))
    assert torch.equal(flat, start)


@pytest.mark.parametrize("sizes", [[0, 1, 31, 64, 200], [512, 0, 513, 0, 0], [0, 0, 0, 0, 7]])
@pytest.mark.parametrize("K,N", [(264, 72), (256, 512)])
def test_grouped(sizes, K, N):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes))
    rows, E = sum(sizes), len(sizes)
    x, dy = (torch.randn(rows, n, generator=g, device="cuda").bfloat16() for n in (K, N))
    offs = torch.tensor([0] + sizes, device="cuda").cumsum(0).to(torch.int32)
    mg = torch.randn(E, K, N, generator=g, device="cuda")
    before = mg.clone()
    ext().grouped_gemm(2, x, dy, offs, mg, True)
    for e in range(E):
        a, b = int(offs[e]), int(offs[e + 1])
        _check(mg[e], before[e], x[a:b], dy[a:b]) if b > a else None
        assert b > a or torch.equal(mg[e], before[e])


@pytest.mark.parametrize("T,splits", [(1, 1), (7, 0), (31, 1), (33, 1), (65, 1), (100, 3), (129, 1), (1000, 0), (1001, 4)])
@pytest.mark.parametrize("M,N", [(8, 264), (264, 512)])
def test_any_token_count(T, splits, M, N):
    g = torch.Generator(device="cuda").manual_seed(T + M)
    dy, x = (torch.full((T + 64, n + 8), float("nan"), device="cuda", dtype=torch.bfloat16) for n in (M, N))
    for t, n in ((dy, M), (x, N)):
        t[:T, :n] = torch.randn(T, n, generator=g, device="cuda")
    dy, x = dy[:T, :M], x[:T, :N]                # NaNs all around
    mg = torch.randn(M, N, generator=g, device="cuda")
    before = mg.clone()
    ext().wgrad_gemm(mg, dy, x, splits, True)
    _check(mg, before, dy, x)


@pytest.mark.parametrize("T,M,N,own", [
    (72, 512, 512, True), (301, 512, 512, True), (328, 512, 512, False),       # few tiles: few tokens only
    (328, 4096, 2048, True), (504, 4096, 2048, True), (520, 4096, 2048, False),            # half of the chip idle
    (1000, 6144, 4096, True), (1001, 6144, 4096, False), (1032, 6144, 4096, False),        # a quarter of the rounds
    (1001, 4096, 4096, True), (3080, 4096, 4096, True), (3071, 4096, 4096, True), (3081, 4096, 4096, False),
    (1000, 8192, 8192, False), (1000, 4096, 2052, False),
])
def test_route_of_ragged_token_counts(T, M, N, own):
    from neuronx_distributed_llama3_2_amd.ops import gemm as G

    g = torch.Generator(device="cuda").manual_seed(T)
    dy, x = (torch.randn(T, n, generator=g, device="cuda").bfloat16() for n in (M, N))
    mg = torch.randn(M, N, generator=g, device="cuda")
    before = mg.clone()
    assert G._use_wgrad_kernel(mg, dy, x) == (own and G._WG_KERNEL != "0")
    if own and G._WG_KERNEL != "0":   # unsplit where the tiles can fill the chip
        assert G._wgrad_kernel_splits(mg, dy, x) == (1 if -(-M // 256) * -(-N // 256) >= 128 else 0)
    G.wgrad_accumulate_(mg, dy, x)
    _check(mg, before, dy, x)


@pytest.mark.parametrize("M,N", [(1272, 4104), (1280, 4104)])   # 20 MB: through the caches below, past them from there on
@pytest.mark.parametrize("T", [96, 100, 1000, 2112])            # both kernels, whole and partial steps
def test_through_and_past_the_caches(M, N, T):
    g = torch.Generator(device="cuda").manual_seed(T + M)
    dy, x = (torch.randn(T, n, generator=g, device="cuda").bfloat16() for n in (M, N))
    whole = torch.randn(M, N + 4, generator=g, device="cuda")
    before = whole.clone()
    print(T, M, N, flush=True)
    ext().wgrad_gemm(whole[:, :N], dy, x, 1, True)
    _check(whole[:, :N], before[:, :N], dy, x)
    assert torch.equal(whole[:, N:], before[:, N:])


@pytest.mark.parametrize("sizes", [[0, 100, 1300], [700, 1, 4000]])   # a mean below and above the line of each
@pytest.mark.parametrize("K,N", [(1288, 1352), (1288, 1360)])         # 20 MB
def test_groups_through_and_past_the_caches(sizes, K, N):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes))
    x, dy = (torch.randn(sum(sizes), n, generator=g, device="cuda").bfloat16() for n in (K, N))
    offs = torch.tensor([0] + sizes, device="cuda").cumsum(0).to(torch.int32)
    mg = torch.randn(len(sizes), K, N, generator=g, device="cuda")
    before = mg.clone()
    print(sizes, K, N, flush=True)
    ext().grouped_gemm(2, x, dy, offs, mg, True)
    for e in range(len(sizes)):
        a, b = int(offs[e]), int(offs[e + 1])
        _check(mg[e], before[e], x[a:b], dy[a:b]) if b > a else None
        assert b > a or torch.equal(mg[e], before[e])
