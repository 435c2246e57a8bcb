"""A product that is first added to a gradient that was just cleared does not read it: when that is so, and what it leaves."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops
from neuronx_distributed_llama3_2_amd.ops.gemm import mark_zero, take_zero, wgrad_accumulate_
from neuronx_distributed_llama3_2_amd.parallel.grad_buffer import FlatBuffer


def _params(device="cpu", shapes=((8, 16), (24, 8))):
    return [torch.nn.Parameter(torch.zeros(s, dtype=torch.bfloat16, device=device)) for s in shapes]


def test_a_mark_is_used_once_and_made_void_by_writes():
    a, b = _params()
    buf = FlatBuffer([a, b])
    assert not take_zero(a.main_grad)   # (nothing was said of it)
    buf.zero_grad()
    assert take_zero(a.main_grad) and not take_zero(a.main_grad)
    for write in (lambda: a.main_grad.add_(1), lambda: buf.grad_data[3:5].fill_(1), lambda: b.main_grad[0].zero_(), buf.finish_grad_sync):
        buf.zero_grad()
        write()
        assert not take_zero(a.main_grad)
    buf.zero_grad()
    a.main_grad = a.main_grad.clone()
    assert not take_zero(a.main_grad) and take_zero(b.main_grad)
    with torch.inference_mode():
        g = torch.zeros(4)
    mark_zero([g])
    assert not take_zero(g)


def test_gradients_that_torch_adds_to():
    a, b = _params()
    buf = FlatBuffer([a, b])
    buf.zero_grad()
    for n in (1, 2):
        (a.float().sum() + 2 * b.float().sum()).backward()
        assert bool((a.main_grad == n).all()) and bool((b.main_grad == 2 * n).all())


@pytest.mark.gpu
@pytest.mark.parametrize("T,M,N", [(64, 512, 264), (1000, 264, 8), (1024, 3328, 3848), (1088, 3328, 3848), (4096, 512, 264), (2100, 4096, 4104)])
def test_dense(T, M, N):
    """Both loops, whole and partial tiles and steps, below and above 20 MB, unsplit and in splits (which add)."""
    g = torch.Generator(device="cuda").manual_seed(T)
    dy, x = (torch.randn(T, n, generator=g, device="cuda").bfloat16() for n in (M, N))
    a, b = torch.zeros(M, N, device="cuda"), torch.zeros(M, N, device="cuda")
    ops.ext().wgrad_gemm(a, dy, x, 1, True)
    ops.ext().wgrad_gemm(b.fill_(float("nan")), dy, x, 1, True, True)   # (not read)
    assert torch.equal(a, b)
    if ops.ext().wgrad_gemm_plan(T, M, N)[0] > 1:
        ops.ext().wgrad_gemm(b.zero_(), dy, x, 0, True, True)
        assert float((a - b).norm()) <= 1e-5 * float(a.norm())   # (fp32 sums in another order)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[100, 0, 37, 200], [1500, 0, 1, 1439], [40] * 4])
@pytest.mark.parametrize("K,N", [(264, 512), (1032, 1288)])
def test_grouped(sizes, K, N):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes))
    x, dy = (torch.randn(sum(sizes), n, generator=g, device="cuda").bfloat16() for n in (K, N))
    offs = torch.tensor([0] + sizes, device="cuda").cumsum(0).to(torch.int32)
    grads = [torch.zeros(len(sizes), K, N, device="cuda") for _ in range(3)]
    grads[2].fill_(float("nan"))
    ops.ext().grouped_gemm(2, x, dy, offs, grads[0], True)
    ops.ext().grouped_gemm(2, x, dy, offs, grads[1], True, True)
    ops.ext().grouped_gemm(2, x, dy, offs, grads[2], False)
    for got in grads[1:]:
        assert float((got - grads[0]).norm()) <= 1e-5 * float(grads[0].norm())
        assert bool((got[[e for e, n in enumerate(sizes) if not n]] == 0).all())


@pytest.mark.gpu
def test_tied_weight_and_micro_batches():
    """The embedding's gradient first, then the head's, twice: the second product of a weight adds, and so does the first after another kernel wrote."""
    g = torch.Generator(device="cuda").manual_seed(5)
    w = torch.nn.Parameter(torch.randn(4096, 4096, generator=g, device="cuda").bfloat16())
    buf = FlatBuffer([w])
    ids = torch.randint(0, 4096, (100,), generator=g, device="cuda")
    dy, x = (torch.randn(100, 4096, generator=g, device="cuda").bfloat16() for _ in range(2))
    want = torch.zeros(4096, 4096, device="cuda", dtype=torch.float64)
    buf.zero_grad()
    for _ in range(2):
        ops.vocab_parallel_embedding(ids, w).backward(x)
        wgrad_accumulate_(w.main_grad, dy, x)
        want.index_add_(0, ids, x.double())
        want += dy.double().t() @ x.double()
    assert float((w.main_grad.double() - want).norm()) < 1e-5 * float(want.norm())


@pytest.mark.gpu
def test_a_recorded_product_reads_what_is_there():
    g = torch.Generator(device="cuda").manual_seed(6)
    w = torch.nn.Parameter(torch.zeros(4096, 4096, device="cuda", dtype=torch.bfloat16))
    buf = FlatBuffer([w])
    dy, x = (torch.randn(100, 4096, generator=g, device="cuda").bfloat16() for _ in range(2))
    once = torch.zeros(4096, 4096, device="cuda")
    wgrad_accumulate_(once, dy, x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        wgrad_accumulate_(w.main_grad, dy, x)
    torch.cuda.current_stream().wait_stream(side)
    buf.zero_grad()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        wgrad_accumulate_(w.main_grad, dy, x)
    for _ in range(2):
        buf.zero_grad()
        graph.replay()
        wgrad_accumulate_(w.main_grad, dy, x)
        graph.replay()
        torch.cuda.synchronize()
        assert float((w.main_grad - 3 * once).norm()) < 1e-5 * float(once.norm())
