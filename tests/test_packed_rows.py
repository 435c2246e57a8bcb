"""How many rows prompts without their padding are given, and when that is done; attention over packed sequences on the CPU."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops
from neuronx_distributed_llama3_2_amd.inference import InferenceConfig
from neuronx_distributed_llama3_2_amd.inference.bucketing import generate_buckets, generated, packed_rows, packing_pays


def test_rows():
    for n in range(1, 20000):
        r = packed_rows(n)
        assert n <= r < n + max(128, n / 8) and r % 128 == 0
    for lo in (1024, 2048, 8192):   # eight row counts for twice the tokens
        assert len({packed_rows(n) for n in range(lo + 1, 2 * lo + 1)}) == 8
    assert not packing_pays(128, 1, 512) and packing_pays(2016, 3, 768) and not packing_pays(2017, 3, 768) and packing_pays(128, 2, 512)


def test_a_list_of_the_callers_own_is_not_packed():
    kw = dict(batch_size=3, seq_len=2048, max_context_length=2048)
    assert generated(InferenceConfig(enable_bucketing=True, **kw))
    assert not generated(InferenceConfig(enable_bucketing=True, buckets=generate_buckets(128, 2048), **kw)) and not generated(InferenceConfig(**kw))


def test_packed_attention_reference():
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(9, h, 8, generator=g) for h in (4, 2, 2))
    o = ops.flash_attn_packed(q, k, v, torch.tensor([0, 2, 2, 8], dtype=torch.int32), 6)
    for a, b in ((0, 2), (2, 8)):
        want = ops.flash_attn_fwd_lse(q[None, a:b], k[None, a:b], v[None, a:b])[0][0]
        assert torch.allclose(o[a:b], want, atol=1e-6)


class _Model:
    def __init__(self):
        self.rows = []

    def forward_packed(self, ids, lengths, slots, rows):
        assert ids.dtype == lengths.dtype == torch.int64 and slots.dtype == torch.int32
        self.rows.append(rows)
        return lengths.float()


def _app(monkeypatch):
    """An application's prefill cache alone; captures are counted."""
    from neuronx_distributed_llama3_2_amd.inference import generation

    captured = []

    def capture(self, device, pool):
        captured.append((*self.shape, self.rows))
        self.graph = type("Graph", (), {"replay": lambda g: None})()
        self.out = self._fwd()

    monkeypatch.setattr(generation.PackedPrefill, "_capture", capture)
    monkeypatch.setattr(torch.cuda, "graph_pool_handle", lambda: (0, 1))
    waits = []
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: waits.append(device))
    app = object.__new__(generation.LlamaForCausalLMInference)
    app.model, app.device, app._prefill_cache, app._prefill_pool = _Model(), torch.device("cpu"), {}, None
    return app, captured, waits


def _ask(app, B, Tb, rows):
    ids = torch.ones(B, Tb, dtype=torch.int32)
    return app._prefill_graph(B, Tb, rows).run(ids, torch.arange(B), torch.full((B,), 4))


def test_a_key_is_captured_when_it_has_come_often(monkeypatch):
    app, captured, _ = _app(monkeypatch)
    for n in range(1, 12):
        assert _ask(app, 3, 768, 1664).tolist() == ([5, 5, 5] if n <= 8 else [0, 0, 0])   # (the stand-in's graph is that of no tokens)
        _ask(app, 3, 768, 1536 - 128 * (n % 4))   # (four others, three times at most)
        assert captured == ([] if n <= 8 else [(3, 768, 1664)])


def test_keys_are_bounded_and_the_oldest_one_goes(monkeypatch):
    from neuronx_distributed_llama3_2_amd.inference.bucketing import PACKED_KEYS

    app, captured, waits = _app(monkeypatch)
    app._prefill_cache[(1, 128)] = "padded"
    for _ in range(9):
        _ask(app, 9, 1024, 1024)
    assert captured == [(9, 1024, 1024)]
    for i in range(PACKED_KEYS - 1):
        _ask(app, 9, 1024, 2048 + 128 * i)
    _ask(app, 9, 1024, 1024)
    _ask(app, 9, 1024, 128)   # (one too many: 2,048 rows were asked for first)
    assert len(app._prefill_cache) == PACKED_KEYS + 1 and (9, 1024, 2048) not in app._prefill_cache and (9, 1024, 1024) in app._prefill_cache
    assert not waits
    for i in range(PACKED_KEYS):
        _ask(app, 9, 2048, 2048 + 128 * i)
    assert len(app._prefill_cache) == PACKED_KEYS + 1 and (9, 1024, 1024) not in app._prefill_cache
    assert len(waits) == 1 and app._prefill_cache[(1, 128)] == "padded"   # (a graph that may run is waited for)


@pytest.mark.parametrize("capturing,mask,rows", [(False, None, 1664), (True, None, 0), (False, "cpu", 1152), (True, "cpu", 0)])
def test_a_call_inside_a_callers_capture_is_not_packed(monkeypatch, capturing, mask, rows):
    app, _, _ = _app(monkeypatch)
    app.config = InferenceConfig(enable_bucketing=True, batch_size=3, seq_len=2048, max_context_length=2048)
    app.model.packed_prefill_ok = lambda: True
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    mask = mask and (torch.arange(540)[None] < torch.tensor([[540], [400], [200]])).long()
    assert app._packed_rows(3, 540, 768, mask) == rows
