"""Products of 17 to 32 rows with a norm, half of the rows a workgroup (csrc/few_rows.hip): halves that differ by a row, one tile to
several a workgroup, groups that are no multiple of 8, both sides of the lines where one workgroup takes all rows again.  Against
64-bit references, with test_few_rows_gpu's bounds; rows past the last stay as they are."""
import pytest
import torch

from test_few_rows_gpu import EPS, PAIR, _close, _exact, _weights

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M", [17, 18, 31, 32])
@pytest.mark.parametrize("N,K", [(8, 64), (1000, 2048), (4096, 1936), (8192, 2048), (8208, 2048), (40, 2064), (3000, 4224), (32784, 2064)])
def test_norm_and_swiglu(M, N, K, int8):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    w, s = _weights(N, K, int8, gen)
    x = (torch.randn(M, K, generator=gen, device="cuda") * 3).bfloat16()
    g = (1 + 0.1 * torch.randn(K, generator=gen, device="cuda")).bfloat16()
    z = _exact(x, g, w, s)
    y = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.ext().dgemv(0, x, g, EPS, w, y[:M], 0, 0, 0, None, None, None, 1, None, None, None, wscale=s)
    _close(y[:M], z)
    assert (y[M] == 7).all()
    h = N // 2
    if h % 4 == 0:
        y = torch.empty(M, h, dtype=torch.bfloat16, device="cuda")
        ops.ext().dgemv(2, x, g, EPS, w, y, 0, 0, 0, None, None, None, 1, None, None, None, wscale=s)
        _close(y, torch.nn.functional.silu(z[:, :h]) * z[:, h:], each=PAIR)


@pytest.mark.parametrize("M,T,nq,nkv,D,H,table", [(17, 1, 8, 2, 64, 2048, True), (30, 2, 32, 8, 64, 2048, False), (31, 1, 4, 4, 128, 4096, True)])
def test_qkv_rope_cache(M, T, nq, nkv, D, H, table):
    import test_few_rows_gpu as F

    F.test_qkv_rope_cache(M, T, nq, nkv, D, H, False, table)
