"""Products with an activation as their epilogue (csrc/act_gemm.hip) against float64: whole tiles, tiles cut into 2 and 4 pieces, ragged rows and
columns, reductions of one step, of half a step and of more steps than the ring holds; and the two sides of the rule that chooses them."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _want(act, x, w):
    """The activation of the product rounded to bf16, and how far a result may be from it."""
    x, w = x.double(), w.double()
    z = x @ w.t()
    # of each product: its rounding to bf16 (2^-8 at most, with its own error in it), the order of the fp32 sums
    dz = z.abs() * 2 ** -8 + (x.abs() @ w.abs().t()) * (x.shape[1] * 2.0 ** -24)
    if act == "relu2":
        y = torch.clamp(z, min=0) ** 2
        dy = 2 * torch.clamp(z, min=0) * dz + dz * dz
    else:
        g, u = z.chunk(2, dim=-1)
        dg, du = dz.chunk(2, dim=-1)
        silu = g * torch.sigmoid(g)
        y = silu * u
        dy = 1.1 * dg * (u.abs() + du) + silu.abs() * du   # |silu'| <= 1.1
    return y, dy + (y.abs() + dy) * 2 ** -8 + 1e-30


@pytest.mark.parametrize("act,R,N,K", [
    ("swiglu", 1, 128, 32), ("relu2", 1, 8, 32), ("swiglu", 65, 256, 96), ("relu2", 257, 136, 160), ("relu2", 129, 264, 64), ("swiglu", 777, 128, 128),
    ("swiglu", 1300, 2048, 192), ("relu2", 1300, 4096, 96),    # 96 tiles, in 2 pieces
    ("swiglu", 2100, 2048, 64), ("relu2", 2200, 4104, 224),    # more, whole
    ("swiglu", 4200, 2048, 256), ("relu2", 4361, 4096, 32),    # a whole round and some more
    ("swiglu", 700, 256, 416), ("relu2", 200, 512, 2080),      # half steps after longer reductions
])
def test_act_gemm(act, R, N, K):
    from neuronx_distributed_llama3_2_amd.ops._ext import gemm_ext

    gen = torch.Generator(device="cuda").manual_seed(R + N + K)
    x = torch.randn(R, K, device="cuda", generator=gen).bfloat16()
    w = torch.randn(N * (2 if act == "swiglu" else 1), K, device="cuda", generator=gen).bfloat16()
    whole = torch.full((R * N + 4096,), 3.0, device="cuda", dtype=torch.bfloat16)   # what lies behind the result stays
    y = whole[: R * N].view(R, N)
    print(act, R, N, K, flush=True)
    gemm_ext().act_gemm({"swiglu": 0, "relu2": 1}[act], x, w, y)
    want, may = _want(act, x, w)
    assert ((y.double() - want).abs() <= may).all()
    assert (whole[R * N:] == 3.0).all()


@pytest.mark.parametrize("act,N,K", [("swiglu", 8192, 2048), ("relu2", 12288, 2048), ("swiglu", 1408, 4096), ("swiglu", 8192, 8192), ("swiglu", 4160, 64)])
def test_rule(act, N, K):
    from neuronx_distributed_llama3_2_amd import ops
    from neuronx_distributed_llama3_2_amd.ops import gemm
    from neuronx_distributed_llama3_2_amd.trace.weight_layout import packed_linear_act

    rows = N * (2 if act == "swiglu" else 1)
    line = -(-192 * 65536 // rows)
    w = (torch.randn(rows, K, device="cuda") * 0.02).bfloat16()
    for R in (line - 1, line):
        x = torch.randn(R, K, device="cuda").bfloat16()
        one = gemm.linear_act(x, w, act)
        assert (one is not None) == (R >= line and K <= 4096 and N % 128 == 0)
        z = gemm.linear(x, w)
        two = ops.swiglu(z) if act == "swiglu" else ops.relu_squared(z)
        got = packed_linear_act(torch.nn.Module(), x, w, None, act)
        assert (got.float() - two.float()).norm() <= 2 ** -7 * two.float().norm()


@pytest.mark.parametrize("act", ["swiglu", "relu2"])
def test_operands_of_other_layouts(act):
    """Rows further apart than they are long, and contiguous operands that begin 8 bytes past a multiple of 16: two launches, either operand alone."""
    from neuronx_distributed_llama3_2_amd.ops import gemm

    R, rows, K = 1024, 16384, 2048
    gen = torch.Generator(device="cuda").manual_seed(1)

    def operands(n):
        flat = torch.randn(n * (K + 32), device="cuda", generator=gen).bfloat16()
        return flat[: n * K].view(n, K), flat.view(n, K + 32)[:, :K], flat[4: 4 + n * K].view(n, K)

    (x, *others), (w, *weights) = operands(R), operands(rows)
    assert gemm.linear_act(x, w, act) is not None
    for a, b in [(o, w) for o in others] + [(x, o) for o in weights]:
        assert gemm.linear_act(a, b, act) is None
