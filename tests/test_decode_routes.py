"""Which kernel a decode product goes to, where the choice can be seen without a GPU."""
import types

import pytest
import torch

from neuronx_distributed_llama3_2_amd.ops import gemv


class _Taken(Exception):
    pass


def _refuse(*_):
    raise _Taken


@pytest.mark.parametrize("rows,stride,dtype,few", [
    (64, 4096, torch.bfloat16, True),
    (18, 2 ** 26, torch.bfloat16, False),      # rows 128 MB apart: past 32-bit offsets, whatever numel says
    (12, 2 ** 27, torch.int8, True),
    (17, 2 ** 27, torch.int8, False),
    (0, 4096, torch.bfloat16, False),
])
def test_rows_far_apart_leave_the_few_rows_kernel(monkeypatch, rows, stride, dtype, few):
    monkeypatch.setattr(gemv, "use_native", lambda *_: True)
    monkeypatch.setattr(gemv, "ext", lambda: types.SimpleNamespace(gemv=_refuse))
    monkeypatch.setattr(gemv, "dequantize_weight", lambda w, s, d: w)
    monkeypatch.setattr(gemv, "_linear", lambda x, w, b: "library")
    w = torch.empty(0, dtype=dtype, device="meta").as_strided((rows, 256), (stride, 1))
    x = torch.empty(9, 256, dtype=torch.bfloat16, device="meta")
    scale = torch.ones(1, device="meta") if dtype == torch.int8 else None
    if few:
        with pytest.raises(_Taken):
            gemv.skinny_linear(x, w, scale)
    else:
        assert gemv.skinny_linear(x, w, scale) == "library"


@pytest.mark.parametrize("tp,rows,width,fused", [
    (2, 8, 4096, True), (2, 8, 4160, False), (2, 7, 4224, True), (2, 9, 2048, False), (2, 32, 2048, False), (2, 3, 8192, True),
    (1, 8, 4160, True), (1, 32, 4224, True), (1, 33, 2048, False),
])
def test_steps_that_are_fused(tp, rows, width, fused):
    """A tensor-parallel step has the limits of csrc/decode_fused.hip (8 rows, 32,768 elements of a norm's rows)."""
    from neuronx_distributed_llama3_2_amd.inference.model_base import DecoderInferenceMixin as Model

    model = types.SimpleNamespace(tp=tp, config=types.SimpleNamespace(hidden_size=width), _decode_fused_ok=True,
                                  _decode_few_ok=width <= 4224, _decode_int8=False)
    ids = types.SimpleNamespace(numel=lambda: rows, is_cuda=True)
    assert Model._decode_fusable(model, ids) is fused


def test_scales_of_int8_weights_are_fp32():
    """Also after a cast of the whole model, which takes the scales along."""
    from neuronx_distributed_llama3_2_amd.inference.model_base import DecoderInferenceMixin as Model
    from neuronx_distributed_llama3_2_amd.quantization.quantization_layers import QuantizedRowParallel

    for kind in ("per_channel_symmetric", "per_tensor_symmetric"):
        mod = QuantizedRowParallel(32, 48, bias=False, quantization_type=kind, quantization_per_channel_axis=0 if "channel" in kind else None)
        mod.quantize_from(torch.randn(48, 32))
        want = mod.scale.reshape(-1)
        for cast in (torch.bfloat16, torch.float32):
            w, scale = Model._weight_scale(mod.to(cast))
            assert w.dtype == torch.int8 and scale.dtype == torch.float32 and scale.is_contiguous()
            assert torch.allclose(scale, want, rtol=2.0 ** -8)


@pytest.mark.parametrize("M,N", [(8, 8), (16384, 2048), (4096, 14336), (64, 4096)])
def test_a_weight_gradient_over_no_tokens_launches_nothing(monkeypatch, M, N):
    from neuronx_distributed_llama3_2_amd.ops import gemm

    def refuse(*_):
        raise AssertionError("launched")

    monkeypatch.setattr(gemm, "_native", lambda *_: True)
    monkeypatch.setattr(gemm, "ext", refuse)
    monkeypatch.setattr(gemm, "gemm_ext", refuse)
    dy, x = (torch.empty(0, n, dtype=torch.bfloat16) for n in (M, N))
    mg = torch.empty(M, N, device="meta")
    gemm.wgrad_accumulate_(mg, dy, x)


@pytest.mark.parametrize("rows,N,K,fused,few", [
    (8, 64, 28672, False, True), (9, 64, 4224, False, True), (16, 128256, 4224, False, True), (9, 64, 4232, False, False),
    (32, 128256, 2048, False, True), (17, 6144, 2056, False, False), (32, 16384, 4096, False, True), (24, 4096, 4096, False, True),
    (25, 4096, 4096, False, False), (32, 8192, 4096, True, True), (32, 8192, 8192, True, False),
])
def test_products_that_stream_their_weights(monkeypatch, rows, N, K, fused, few):
    """9 to 32 rows go to csrc/few_rows.hip only where that is the faster product, in the op and in the unfused step."""
    from neuronx_distributed_llama3_2_amd.inference import model_base

    assert gemv.few_rows_pay(rows, N, K, fused) is few
    monkeypatch.setattr(gemv, "use_native", lambda *_: True)
    monkeypatch.setattr(gemv, "ext", lambda: types.SimpleNamespace(gemv=_refuse))
    monkeypatch.setattr(gemv, "_linear", lambda x, w, b: torch.empty(x.shape[0], w.shape[0], device="meta"))
    mod = types.SimpleNamespace(weight=torch.empty(N, K, dtype=torch.bfloat16, device="meta"), bias=None)
    x = torch.empty(rows, K, dtype=torch.bfloat16, device="meta")
    if few:
        with pytest.raises(_Taken):
            gemv.skinny_linear(x, mod.weight, glu=fused)
    else:
        monkeypatch.setattr("neuronx_distributed_llama3_2_amd.ops.activations.swiglu", lambda y: y)
        assert gemv.skinny_linear(x, mod.weight, glu=fused).shape == (rows, N)
    taken = []
    monkeypatch.setattr(model_base, "skinny_linear", lambda *a, **k: taken.append(1))
    monkeypatch.setattr("neuronx_distributed_llama3_2_amd.trace.weight_layout.packed_linear", lambda *a: x)
    monkeypatch.setattr(model_base.ops, "swiglu", lambda y: y)
    on_gpu = type("X", (), {"is_cuda": True, "dtype": torch.bfloat16, "shape": (rows, K), "numel": lambda self: rows * K})()
    model_base.DecoderInferenceMixin._proj(mod, on_gpu, glu=fused)
    assert bool(taken) is few


@pytest.mark.parametrize("rows,N,K,fused,few", [
    (16, 12288, 8192, False, True), (17, 8192, 8192, False, True), (32, 8200, 8192, False, False), (32, 8192, 3072, False, False),
    (32, 8192, 3072, True, True), (17, 2048, 2048, False, True),
])
def test_hybrid_projections_that_stream_their_weights(rows, N, K, fused, few):
    from neuronx_distributed_llama3_2_amd.modules.hybrid.context import streams

    assert streams(rows, N, K, fused) is few
