"""Products are added to what a gradient holds, whoever wrote it since it was cleared and by whatever way: torch's count of writes does not see them all."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops
from neuronx_distributed_llama3_2_amd.ops.gemm import wgrad_accumulate_
from neuronx_distributed_llama3_2_amd.parallel.grad_buffer import FlatBuffer


def test_gradients_that_torch_adds_to():
    a, b = (torch.nn.Parameter(torch.zeros(s, dtype=torch.bfloat16)) for s in ((8, 16), (24, 8)))
    buf = FlatBuffer([a, b])
    buf.zero_grad()
    for n in (1, 2):
        (a.float().sum() + 2 * b.float().sum()).backward()
        assert bool((a.main_grad == n).all()) and bool((b.main_grad == 2 * n).all())


def _buffer(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.nn.Parameter(torch.randn(4096, 4096, generator=g, device="cuda").bfloat16())
    dy, x = (torch.randn(100, 4096, generator=g, device="cuda").bfloat16() for _ in range(2))
    return w, FlatBuffer([w]), dy, x


def _close(got, want):
    assert float((got.double() - want.double()).norm()) < 1e-5 * float(want.double().norm())   # (fp32 sums in another order)


@pytest.mark.gpu
@pytest.mark.parametrize("write", ["data", "kernel", "alias"])
def test_what_is_written_after_clearing_is_added_to(write):
    """Restored sums, a caller's own kernel, an alias taken before: none of them moves the gradient's version."""
    w, buf, dy, x = _buffer(4)
    once = torch.zeros(4096, 4096, device="cuda")
    wgrad_accumulate_(once, dy, x)
    saved = torch.randn(4096, 4096, device="cuda")
    before = w.main_grad.data
    buf.zero_grad()
    if write == "data":
        w.main_grad.data.copy_(saved)
    elif write == "kernel":
        ops.ext().wgrad_gemm(w.main_grad, dy, x, 1, True)
        saved = once
    else:
        before.add_(saved)
    wgrad_accumulate_(w.main_grad, dy, x)
    _close(w.main_grad, saved + once)


@pytest.mark.gpu
def test_tied_weight_and_micro_batches():
    """The embedding's gradient first, then the head's, twice."""
    w, buf, dy, x = _buffer(5)
    g = torch.Generator(device="cuda").manual_seed(5)
    ids = torch.randint(0, 4096, (100,), generator=g, device="cuda")
    want = torch.zeros(4096, 4096, device="cuda", dtype=torch.float64)
    buf.zero_grad()
    for _ in range(2):
        ops.vocab_parallel_embedding(ids, w).backward(x)
        wgrad_accumulate_(w.main_grad, dy, x)
        want.index_add_(0, ids, x.double())
        want += dy.double().t() @ x.double()
    _close(w.main_grad, want)


@pytest.mark.gpu
@pytest.mark.parametrize("recorded", ["product", "torch"])
def test_a_replay_is_added_to(recorded):
    """A product, or torch's addition of a .grad, recorded into a graph, and an eager product after its replay."""
    w, buf, dy, x = _buffer(6)
    once, add = torch.zeros(4096, 4096, device="cuda"), torch.randn(4096, 4096, device="cuda").bfloat16()
    wgrad_accumulate_(once, dy, x)

    def work():
        if recorded == "product":
            wgrad_accumulate_(w.main_grad, dy, x)
        else:
            (w * 1.0).backward(add)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        work()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    buf.zero_grad()
    with torch.cuda.graph(graph):
        work()
    part = once if recorded == "product" else add.float()
    for _ in range(2):
        buf.zero_grad()
        graph.replay()
        wgrad_accumulate_(w.main_grad, dy, x)
        graph.replay()
        torch.cuda.synchronize()
        _close(w.main_grad, once + 2 * part)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[100, 0, 37, 200], [1500, 0, 1, 1439], [40] * 4])
@pytest.mark.parametrize("K,N", [(264, 512), (1032, 1288)])
def test_groups_gradients_that_the_call_clears(sizes, K, N):
    """accumulate=False: the call clears the gradients itself, and its products do not read them."""
    g = torch.Generator(device="cuda").manual_seed(sum(sizes))
    x, dy = (torch.randn(sum(sizes), n, generator=g, device="cuda").bfloat16() for n in (K, N))
    offs = torch.tensor([0] + sizes, device="cuda").cumsum(0).to(torch.int32)
    added, own = torch.zeros(len(sizes), K, N, device="cuda"), torch.full((len(sizes), K, N), float("nan"), device="cuda")
    ops.ext().grouped_gemm(2, x, dy, offs, added, True)
    ops.ext().grouped_gemm(2, x, dy, offs, own, False)
    _close(own, added)
    assert bool((own[[e for e, n in enumerate(sizes) if not n]] == 0).all())
