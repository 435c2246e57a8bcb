"""Products with an activation whose workgroups have several tiles (csrc/act_gemm.hip): two to five rounds of the CUs, reductions of 2, 3 and more steps, where
the loads go over to the next tile at once, after one step or later, rows and columns that fill no tile (whose stores are not counted), and rounds that end in
pieces.  Against float64, with the bounds of test_act_gemm_gpu.py."""

import pytest
import torch
from test_act_gemm_gpu import _want

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act,R,N,K", [
    ("relu2", 4361, 8200, 128), ("relu2", 4361, 8200, 192), ("relu2", 4096, 8192, 256), ("relu2", 5000, 8192, 320),     # two rounds and some
    ("swiglu", 6000, 4096, 128), ("swiglu", 6100, 4096, 192), ("swiglu", 4352, 4224, 448),                              # three, two and pieces
    ("relu2", 10240, 8192, 128), ("swiglu", 10300, 4096, 192),                                                          # five: a run of four and one more
])
def test_runs(act, R, N, K):
    from neuronx_distributed_llama3_2_amd.ops._ext import gemm_ext

    gen = torch.Generator(device="cuda").manual_seed(R + N + K)
    x = torch.randn(R, K, device="cuda", generator=gen).bfloat16()
    w = torch.randn(N * (2 if act == "swiglu" else 1), K, device="cuda", generator=gen).bfloat16()
    whole = torch.full((R * N + 4096,), 3.0, device="cuda", dtype=torch.bfloat16)
    y = whole[: R * N].view(R, N)
    print(act, R, N, K, flush=True)
    for _ in range(2):
        gemm_ext().act_gemm({"swiglu": 0, "relu2": 1}[act], x, w, y)
        for r in range(0, R, 1024):   # (float64, some rows at a time)
            want, may = _want(act, x[r:r + 1024], w)
            assert ((y[r:r + 1024].double() - want).abs() <= may).all()
        assert (whole[R * N:] == 3.0).all()
        y.fill_(float("nan"))
