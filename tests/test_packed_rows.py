"""How many rows prompts without their padding are given, and when that is done; attention over packed sequences on the CPU."""
import torch

from neuronx_distributed_llama3_2_amd import ops
from neuronx_distributed_llama3_2_amd.inference import InferenceConfig
from neuronx_distributed_llama3_2_amd.inference.bucketing import generate_buckets, generated, packed_rows, packing_pays


def test_rows():
    for n in range(1, 20000):
        r = packed_rows(n)
        assert n <= r < n + max(128, n / 8) and r % 128 == 0
    for lo in (1024, 2048, 8192):   # at most eight graphs for twice the tokens
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
