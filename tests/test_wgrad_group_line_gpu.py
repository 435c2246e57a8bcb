"""Groups' weight gradients on both sides of the mean count of tokens from which the tile loop takes gradients of 20 MB and more, with groups that are empty,
short, and no multiple of a step."""
import pytest
import torch

from test_wgrad_tiles_gpu import _among_nans, _check

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[900] * 4, [901] * 4, [0, 1, 2163, 1440], [905, 0, 2699, 0], [63, 65, 1727, 1745]])
def test_groups(sizes):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes))
    E, K, N, rows = len(sizes), 1032, 1288, sum(sizes)
    x, dy = _among_nans(rows, K, g), _among_nans(rows, N, g)
    offs = torch.tensor([0] + sizes, device="cuda").cumsum(0).to(torch.int32)
    mg = torch.randn(E, K, N, generator=g, device="cuda")
    before = mg.clone()
    ops.ext().grouped_gemm(2, x.contiguous(), dy.contiguous(), offs, mg, True)
    for e in range(E):
        a, b = int(offs[e]), int(offs[e + 1])
        if b > a:
            _check(mg[e], before[e], x[a:b], dy[a:b])
        else:
            assert torch.equal(mg[e], before[e])
