"""Products of 1 to 32 rows (csrc/few_rows.hip) against 64-bit references: edges of the tiles of rows, weight rows and
reduction chunks, every geometry of the dispatch, both weight types and all epilogues.

Tolerance: outputs and x times the norm's weight are rounded to bf16 (relative error of at most 2^-9 each, 2^-9 / sqrt(3)
on average), sums are fp32: 2-norm within 3 x 2^-9 of the reference; the rotary epilogue rounds twice.  Single values: two
roundings of the result (2^-8 of it), and of a sum's operands (2^-9 / sqrt(3) of the values' root mean square, at random: 14
standard deviations are 8 x 2^-9); products of two sums err with either factor times the other, up to 5.5 times its root mean
square: 2 x 5.5 x 8 x 2^-9 of the squared root mean square, which is 2 to 3 times the products' own."""

import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu
TOL = 3 * 2 ** -9
EPS = 1e-5


def _weights(N, K, int8, gen):
    if int8:
        return (torch.randint(-128, 128, (N, K), generator=gen, device="cuda", dtype=torch.int8),
                torch.rand(N, generator=gen, device="cuda") * 3e-4 + 1e-5)
    return (torch.randn(N, K, generator=gen, device="cuda") * 0.02).bfloat16(), None


def _exact(x, norm, w, scale):
    x = x.double()
    if norm is not None:
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * norm.double()
    return x @ (w.double() if scale is None else w.double() * scale.double()[:, None]).t()


PAIR = 2 ** -1   # (single values of SwiGLU and the squared ReLU)


def _close(got, want, tol=TOL, each=None):
    err = (got.double() - want).abs()
    assert torch.isfinite(got.float()).all() and float(err.norm() / want.norm()) < tol
    rms = float(want.square().mean().sqrt())
    assert (err <= (2 ** -8 if tol >= TOL else 8 * tol) * want.abs() + (8 / 3 * tol if each is None else each) * rms).all(), float(err.max()) / rms


SHAPES = [(1, 64, 128), (3, 40, 8), (3, 100, 136), (16, 1000, 2048), (17, 3072, 2048), (32, 4112, 2048), (5, 2048, 2048),
          (32, 6144, 4096), (13, 4096, 4096), (29, 40, 4224), (16, 4096, 1920)]
LONG = [(4, 2048, 8192), (9, 2048, 8192), (32, 100, 5000), (13, 4096, 14336), (17, 4096, 4352), (16, 33, 4240)]


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES + LONG)
def test_store_and_residual(M, N, K, int8):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    if int8 and K % 16:
        K += 8
    w, s = _weights(N, K, int8, gen)
    M = M if int8 else max(M, 3)
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    y0 = torch.randn(M, N, generator=gen, device="cuda").bfloat16()
    want = _exact(x, None, w, s)
    C = ops.ext()
    tickets = torch.zeros(256, dtype=torch.int32, device="cuda")
    outs = []
    for _ in range(2):   # (the counters are left as they were, and the order of the sums does not change)
        y = y0.clone()
        C.dgemv(1, x, None, 0.0, w, y, 0, 0, 0, None, None, None, 1, None, None, None, wscale=s, tickets=tickets)
        outs.append(y)
    _close(outs[0], y0.double() + want)
    assert torch.equal(outs[0], outs[1]) and not tickets.any()
    y = torch.empty_like(y0)
    C.dgemv(0, x, None, 0.0, w, y, 0, 0, 0, None, None, None, 1, None, None, None, wscale=s)
    _close(y, want)
    if not int8:
        yf = torch.empty(M, N, device="cuda")
        C.dgemv(0, x, None, 0.0, w, yf, 0, 0, 0, None, None, None, 1, None, None, None)
        _close(yf, want, 1e-5)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_norm_and_swiglu(M, N, K, int8):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K + 1)
    if int8 and K % 16:
        K += 8
    M = M if int8 else max(M, 3)
    w, s = _weights(2 * N, K, int8, gen)
    x = (torch.randn(M, K, generator=gen, device="cuda") * 3).bfloat16()
    g = (1 + 0.1 * torch.randn(K, generator=gen, device="cuda")).bfloat16()
    z = _exact(x, g, w, s)
    C = ops.ext()
    y = torch.empty(M, 2 * N, dtype=torch.bfloat16, device="cuda")
    C.dgemv(0, x, g, EPS, w, y, 0, 0, 0, None, None, None, 1, None, None, None, wscale=s)
    _close(y, z)
    y = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    C.dgemv(2, x, g, EPS, w, y, 0, 0, 0, None, None, None, 1, None, None, None, wscale=s)
    _close(y, torch.nn.functional.silu(z[:, :N]) * z[:, N:], each=PAIR)


@pytest.mark.parametrize("M,T,nq,nkv,D,H,int8,table", [(3, 1, 4, 2, 64, 512, False, True), (8, 2, 8, 2, 64, 2048, False, False),
                                                       (32, 1, 32, 8, 64, 2048, False, True), (18, 3, 8, 8, 128, 4096, False, True),
                                                       (6, 1, 6, 2, 32, 144, True, False), (20, 4, 48, 8, 128, 4096, True, True)])
def test_qkv_rope_cache(M, T, nq, nkv, D, H, int8, table):
    gen = torch.Generator(device="cuda").manual_seed(M * D)
    N, Lmax, B = (nq + 2 * nkv) * D, 64, M // T
    w, s = _weights(N, H, int8, gen)
    g = (1 + 0.1 * torch.randn(H, generator=gen, device="cuda")).bfloat16()
    rows = torch.randn(50, H, generator=gen, device="cuda").bfloat16()
    ids = torch.randint(0, 50, (M,), generator=gen, device="cuda")
    pos = torch.arange(M, device="cuda") * 5 % (Lmax + 9)   # (some past the cache's end: not written)
    if table:
        ids[0] = -1                                         # (not a row of the table: zeros)
    x = rows[ids.clamp(min=0)] * (ids >= 0)[:, None]
    ang = torch.rand(Lmax + 9, D // 2, generator=gen, device="cuda") * 6
    cos, sin = ang.cos(), ang.sin()
    idx = torch.randperm(B, generator=gen, device="cuda").to(torch.int32)
    kc, vc = (torch.zeros(B, nkv, Lmax, D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    y, copy = torch.empty(M, N, dtype=torch.bfloat16, device="cuda"), torch.full((M, H), 7.0, device="cuda").bfloat16()
    kw = dict(xidx=ids, xcopy=copy) if table else {}
    ops.ext().dgemv(3, rows if table else x.contiguous(), g, EPS, w, y, nq, nkv, D, cos, sin, pos, T, kc, vc, idx, wscale=s, **kw)
    if table:
        assert torch.equal(copy, x)
    z = _exact(x, g, w, s).view(M, nq + 2 * nkv, D)
    c, si = cos[pos].double()[:, None], sin[pos].double()[:, None]
    a, b = z[:, :nq + nkv].chunk(2, -1)
    want = torch.cat([torch.cat([a * c - b * si, b * c + a * si], -1), z[:, nq + nkv:]], 1)
    _close(y.view(M, -1, D), want, 2 * TOL)
    for m in range(M):
        if pos[m] < Lmax:
            slot = int(idx[m // T])
            assert torch.equal(kc[slot, :, pos[m]], y.view(M, -1, D)[m, nq:nq + nkv])
            assert torch.equal(vc[slot, :, pos[m]], y.view(M, -1, D)[m, nq + nkv:])


@pytest.mark.parametrize("M,N,K", [(3, 48, 64), (16, 12288, 2048), (32, 2064, 1024), (17, 2048, 12288)])
def test_linear_few_epilogues(M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    w, _ = _weights(N, K, False, gen)
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    z = _exact(x, None, w, None)
    tickets = torch.zeros(ops.experts.LINEAR_TICKETS, dtype=torch.int32, device="cuda")
    _close(ops.linear_few(x, w, tickets=tickets), z)
    assert not tickets.any()
    _close(ops.linear_few(x, w, "relu2"), z.clamp(min=0).square(), each=PAIR)
    _close(ops.linear_few(x, w, "f32", alpha=0.5), 0.5 * z, 1e-5)
    _close(ops.linear_few(x, w, "f32", alpha=0.5, cap=0.3), 0.3 * torch.tanh(0.5 * z / 0.3), 1e-5)


def test_rows_of_a_view_and_unaligned_outputs():
    """Inputs between other columns; outputs whose rows start at odd places."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    w, _ = _weights(51, 256, False, gen)
    x = torch.randn(7, 512, generator=gen, device="cuda").bfloat16()[:, 128:384]
    y = torch.zeros(7, 53, dtype=torch.bfloat16, device="cuda")
    ops.ext().dgemv(0, x, None, 0.0, w, y[:, 1:52], 0, 0, 0, None, None, None, 1, None, None, None)
    _close(y[:, 1:52], _exact(x, None, w, None))
    assert not y[:, 0].any() and not y[:, 52].any()


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (12, 40, 4368), (13, 2048, 9216), (9, 24, 9232), (9, 2048, 12288),            # up to 128 tiles, both lengths of parts
    (12, 4096, 12432), (17, 2064, 4368), (32, 4096, 11008), (19, 8200, 14336),    # more of them, two tiles of rows
])
def test_split_reductions(M, N, K, int8):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    w, s = _weights(N, K, int8, gen)
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    y0 = torch.randn(M, N, generator=gen, device="cuda").bfloat16()
    want = _exact(x, None, w, s)
    need = ops.ext().few_rows_tickets(M, N, K)
    assert need > 0 and (need <= 1024 or N > 8192)   # (it is split; the models' counters serve up to 8,192 weight rows)
    tickets = torch.zeros(need + 2, dtype=torch.int32, device="cuda")
    run = lambda y, e, t: ops.ext().dgemv(e, x, None, 0.0, w, y, 0, 0, 0, None, None, None, 1, None, None, None, wscale=s, tickets=t)
    outs = []
    for t in (tickets[:need], tickets[:need], tickets[:need - 1]):   # (too few counters: not split)
        y = y0.clone()
        run(y, 1, t)
        outs.append(y)
        _close(y, y0.double() + want)
    assert torch.equal(outs[0], outs[1]) and not tickets.any()
    graph = torch.cuda.CUDAGraph()
    y = y0.clone()
    with torch.cuda.graph(graph):
        run(y, 1, tickets[:need])
    for _ in range(3):
        y.copy_(y0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, outs[0]) and not tickets.any()


@pytest.mark.parametrize("M", [17, 20, 31, 32])
@pytest.mark.parametrize("N,K", [(8, 64), (1000, 4224), (2048, 2048), (2049, 136)])   # (the last: both halves by one workgroup)
def test_rows_in_two_halves(M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    w, _ = _weights(N, K, False, gen)
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    z = _exact(x, None, w, None)
    _close(ops.linear_few(x, w), z)
    _close(ops.linear_few(x, w, "relu2"), z.clamp(min=0).square(), each=PAIR)
    _close(ops.linear_few(x, w, "f32", alpha=0.5, cap=0.3), 0.3 * torch.tanh(0.5 * z / 0.3), 1e-5)
