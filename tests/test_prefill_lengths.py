"""Lengths that prompts are padded to, and that the logits do not depend on them."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd.inference import InferenceConfig
from neuronx_distributed_llama3_2_amd.inference.bucketing import pad_to_bucket, prefill_lengths


@pytest.mark.parametrize("batch,top,given,want", [
    (1, 2048, None, [128, 256, 512, 768, 1024, 1536, 2048]),
    (3, 2048, None, [128, 256, 384, 512, 768, 1024, 1536, 2048]),
    (8, 512, None, [128, 192, 256, 384, 512]),
    (1, 1100, None, [128, 256, 512, 768, 1100]),            # the last bucket is no power of two
    (64, 128, None, [128]), (64, 100, None, [100]),
    (3, 2048, [128, 1024, 2048], [128, 1024, 2048]),        # a caller's own
])
def test_lengths(batch, top, given, want):
    cfg = InferenceConfig(batch_size=batch, seq_len=4096, max_context_length=top, enable_bucketing=True, buckets=given)
    kept = list(cfg.buckets)
    assert sorted(prefill_lengths(cfg, batch)) == want + [4096] and cfg.buckets == kept
    plain = InferenceConfig(batch_size=batch, seq_len=4096, max_context_length=top)
    assert prefill_lengths(plain, batch) == [top, 4096]
    assert prefill_lengths(cfg, batch, False) == kept + [4096]
    for T in range(1, 4097, 61):   # never longer than the bucket, and what none holds is refused as before
        ids = torch.zeros((1, T), dtype=torch.long)
        n = pad_to_bucket(ids, ids, prefill_lengths(cfg, batch), 0)[0].shape[1]
        assert T <= n <= min(b for b in kept + [4096] if b >= T)
    with pytest.raises(ValueError):
        pad_to_bucket(torch.zeros((1, 4097)), torch.zeros((1, 4097)), prefill_lengths(cfg, batch), 0)


def test_a_list_of_the_callers_own_stands(tmp_path):
    """Also where it is the one that would have been generated, and after saving; files from before the list's origin was kept in
    them hold a list."""
    import json

    kw = dict(batch_size=3, seq_len=2048, max_context_length=1024, enable_bucketing=True)
    made = InferenceConfig(**kw)
    own = InferenceConfig(buckets=[128, 256, 512, 1024], **kw)
    assert made.buckets == own.buckets
    for cfg, more in ((made, [384, 768]), (own, [])):
        cfg.save_pretrained(str(tmp_path))
        for c in (cfg, InferenceConfig.from_pretrained(str(tmp_path))):
            assert sorted(prefill_lengths(c, 3)) == sorted([128, 256, 512, 1024, 2048] + more)
    made.save_pretrained(str(tmp_path))
    path = tmp_path / "nxd_inference_config.json"
    kept = json.loads(path.read_text())
    del kept["buckets_generated"]
    path.write_text(json.dumps(kept))
    assert prefill_lengths(InferenceConfig.from_pretrained(str(tmp_path)), 3) == [128, 256, 512, 1024, 2048]


def test_logits_do_not_depend_on_the_length():
    from test_inference import _hf_model, _tiny_cfg
    from neuronx_distributed_llama3_2_amd.inference import LlamaForCausalLMInference
    from neuronx_distributed_llama3_2_amd.models.llama.convert import hf_to_nxd

    cfg = _tiny_cfg(max_position_embeddings=512)
    sd = _hf_model(cfg).state_dict()
    models = []
    for buckets in (None, [128, 256, 512]):
        icfg = InferenceConfig(batch_size=4, seq_len=512, max_context_length=512, enable_bucketing=True, buckets=buckets)
        icfg.enable_bucketing = buckets is None
        models.append(LlamaForCausalLMInference(cfg, icfg, dtype=torch.float32, init_weights=False))
        models[-1]._load_full(hf_to_nxd(sd, cfg))
    torch.manual_seed(7)
    ids = torch.randint(3, cfg.vocab_size, (4, 150))
    mask = (torch.arange(150)[None] < torch.tensor([150, 131, 128, 1])[:, None]).long()
    a, b = (m._context_encode(ids, mask) for m in models)   # padded to 192 and to 256
    torch.testing.assert_close(a, b, atol=1e-5, rtol=1e-5)
    a, b = (m.generate(ids[:, :140], max_new_tokens=6, eos_token_id=-1) for m in models)
    assert torch.equal(a, b)
