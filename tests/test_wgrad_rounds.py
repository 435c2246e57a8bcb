"""Weight gradients that fill their rounds of 256 tiles go to csrc/wgrad_gemm.hip, whatever the tokens, and nobody writes transposed copies for them.  The lines
were measured (ops/gemm.py); the gradients are compared with float64."""
import pytest
import torch

from test_wgrad_tiles_gpu import _check

from neuronx_distributed_llama3_2_amd import ops
from neuronx_distributed_llama3_2_amd.ops import gemm


@pytest.mark.parametrize("T,M,N,own", [
    (3072, 4096, 4096, True), (3008, 4096, 4096, False), (3009, 4096, 4096, True), (1, 4096, 4096, True), (2048, 16384, 16384, False),   # tokens
    (3072, 4096, 3584, True), (3072, 4096, 3328, False), (3072, 4096, 5504, True), (3072, 4096, 5376, False), (3001, 4096, 5376, False),     # fill: 224, 208, 352, 336 tiles
    (3072, 8192, 5376, True), (3072, 8192, 5120 + 256 * 3 + 8, True), (3001, 4096, 4092, False), (3001, 4100, 4096, False),
])
def test_rule(T, M, N, own):
    assert gemm.wgrad_in_rounds(T, M, N) == (own and gemm._WG_KERNEL != "0")


@pytest.mark.gpu
@pytest.mark.parametrize("T,M,N", [(3072, 4096, 3592), (3009, 3592, 4096), (1, 4096, 4096), (72, 5640, 4096), (4100, 4096, 4096), (3079, 5632, 4096)])
@pytest.mark.parametrize("copy", [False, True])
def test_gradient(T, M, N, copy):
    g = torch.Generator(device="cuda").manual_seed(T + M)
    dy, x = (torch.randn(T, n, generator=g, device="cuda").bfloat16() for n in (M, N))
    mg = torch.randn(M, N, generator=g, device="cuda")
    before = mg.clone()
    assert gemm._use_wgrad_in_rounds(mg, dy, x) == gemm.wgrad_in_rounds(T, M, N)
    gemm.wgrad_accumulate_(mg, dy, x, go_t=dy.t().contiguous() if copy else None)
    _check(mg, before, dy, x)


@pytest.mark.gpu
def test_operands_that_the_kernel_does_not_take():
    g = torch.Generator(device="cuda").manual_seed(1)
    dy, x = (torch.randn(100, 4104, generator=g, device="cuda").bfloat16() for _ in range(2))
    mg = torch.zeros(4096, 4096, device="cuda")
    assert gemm._use_wgrad_in_rounds(mg, dy[:, :4096], x[:, 8:]) == (gemm._WG_KERNEL != "0")
    for a, b in ((dy[:, 4:4100], x[:, 8:]), (dy[:, 8:], x[:, 4:4100]), (dy[:, :4096], x[:, 8:].half()), (dy[:, :4096], None)):
        assert not gemm._use_wgrad_in_rounds(mg, a, b)
    assert not gemm._use_wgrad_in_rounds(mg.bfloat16(), dy[:, :4096], x[:, 8:])


@pytest.mark.gpu
@pytest.mark.parametrize("rows,width,copies", [(3072, 4096, False), (3008, 4096, True), (3072, None, True)])
def test_swiglu_writes_copies_for_the_library_only(rows, width, copies):
    g = torch.Generator(device="cuda").manual_seed(rows)
    gu = torch.randn(rows, 8192, generator=g, device="cuda").bfloat16()
    dh = torch.randn(rows, 4096, generator=g, device="cuda").bfloat16()
    seen, out = [], []
    for token_major in (True, False):
        leaf = gu.clone().requires_grad_()
        leaf.register_hook(lambda d: seen.append(hasattr(d, "_nxd_t")))
        h = ops.swiglu(leaf, token_major=token_major, width=width)
        assert hasattr(h, "_nxd_t") == (copies and token_major)
        h.backward(dh)
        out.append((h.detach(), leaf.grad))
    assert seen == [copies, False]
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("name,value", [("_WGRAD_BF16", True), ("_WGRAD_T", "2"), ("_WG_KERNEL", "0")])
def test_switches_that_ask_for_the_library(name, value, monkeypatch):
    monkeypatch.setattr(gemm, name, value)
    assert not gemm.wgrad_in_rounds(8192, 4096, 4096)


@pytest.mark.gpu
def test_a_gradient_that_is_asked_for_in_16_bits(monkeypatch):
    """NXD_WGRAD_BF16=1: what a producer's copies come with is rounded to bf16 before it is added to the fp32 gradient."""
    monkeypatch.setattr(gemm, "_WGRAD_BF16", True)
    g = torch.Generator(device="cuda").manual_seed(2)
    dy, x = torch.randn(4096, 8192, generator=g, device="cuda").bfloat16(), torch.randn(4096, 8192, generator=g, device="cuda").bfloat16()
    mg = torch.zeros(8192, 8192, device="cuda")
    gemm.wgrad_accumulate_(mg, dy, x, go_t=dy.t().contiguous())
    assert torch.equal(mg, mg.bfloat16().float())
    want = dy.double().t() @ x.double()
    assert float((mg.double() - want).norm()) < 2 ** -8 * float(want.norm())


def _mlp(width, inter, device, grad_dtype):
    """A Llama MLP and what its SwiGLU was told of the width; grad_dtype: of its gradient buffer, None: it has none."""
    from neuronx_distributed_llama3_2_amd.models.llama.modeling_llama import LlamaMLP, llama_config
    from neuronx_distributed_llama3_2_amd.parallel.grad_buffer import FlatBuffer
    from neuronx_distributed_llama3_2_amd.parallel_layers import parallel_state as ps
    import torch.distributed as dist

    if not dist.is_initialized():
        dist.init_process_group("gloo", store=dist.HashStore(), rank=0, world_size=1)
    if not ps.model_parallel_is_initialized():
        ps.initialize_model_parallel(1)
    mlp = LlamaMLP(llama_config("tiny", hidden_size=width, intermediate_size=inter), torch.bfloat16, torch.device(device))
    buf = FlatBuffer(list(mlp.parameters()), grad_dtype=grad_dtype) if grad_dtype is not None else None
    return mlp, buf


@pytest.mark.parametrize("grad_dtype,width", [(torch.float32, 64), (torch.bfloat16, None), (None, None)])
def test_swiglu_is_told_the_width_where_the_kernel_can_add_to_the_gradients(grad_dtype, width, monkeypatch):
    from neuronx_distributed_llama3_2_amd.models.llama import modeling_llama

    mlp, _ = _mlp(64, 128, "cpu", grad_dtype)
    told = []
    monkeypatch.setattr(modeling_llama.ops, "swiglu", lambda gu, token_major=False, width=None: told.append(width) or ops.swiglu_reference(gu))
    for selective in (False, True):
        mlp.selective_checkpoint = selective
        mlp(torch.randn(5, 1, 64).bfloat16().requires_grad_())
    assert told == [width, width]


@pytest.mark.gpu
@pytest.mark.parametrize("grad_dtype", [torch.float32, torch.bfloat16, None])
def test_an_mlp_whose_gradients_go_to_the_library_has_its_copies(grad_dtype):
    """3,072 tokens, 4096 wide, 3840: both gradients fill their rounds of tiles.  Against float64; a 16-bit gradient is rounded once more (2^-9)."""
    mlp, buf = _mlp(4096, 3840, "cuda", grad_dtype)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(3072, 1, 4096, generator=g, device="cuda").bfloat16().requires_grad_()
    gu = mlp.gate_up_proj(x)
    h = mlp.act(gu, 4096)
    assert hasattr(h, "_nxd_t") == (grad_dtype is not torch.float32)
    dy = torch.randn(3072, 1, 4096, generator=g, device="cuda").bfloat16()
    if buf is not None:
        buf.zero_grad()
    mlp.down_proj(h).backward(dy)
    w = mlp.down_proj.weight
    got = w.main_grad if buf is not None else w.grad
    want = dy[:, 0].double().t() @ h[:, 0].double()
    assert float((got.double() - want).norm()) < (1e-5 if grad_dtype is torch.float32 else 3 * 2 ** -9) * float(want.norm())
