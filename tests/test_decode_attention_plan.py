"""How decode attention shares the keys of a sequence out to key splits: every length is covered within the caller's partial
buffers, by the sequence's own length whatever the cache has room for, in so few splits that adding them up stays short."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops


def _plan(*a, tickets=True):
    return ops.ext().decode_attn_plan(*a, tickets)


@pytest.mark.parametrize("tickets", [False, True])
@pytest.mark.parametrize("M,D", [(1, 64), (4, 64), (4, 128), (16, 64), (16, 128)])
@pytest.mark.parametrize("heads", [(1, 1), (1, 8), (3, 2), (13, 8), (64, 8)])
@pytest.mark.parametrize("room", [1, 100, 128, 129, 1024, 2304, 8192, 32768, 65537, 131072])
def test_every_length_is_covered(room, heads, M, D, tickets):
    splits, _, merges = _plan(room, *heads, M, D, room, tickets=tickets)
    assert tickets or not merges
    assert splits <= -(-room // 128)
    for n in {0, 1, 63, 127, 128, 129, room // 3, room // 2, room - 1, room} & set(range(room + 1)):
        s, keys, _ = _plan(room, *heads, M, D, n, tickets=tickets)
        assert s == splits and keys % 64 == 0 and keys >= 128 and splits * keys >= n
        live = -(-n // keys)
        if keys < 1024:
            assert live <= (16 if M * D > 256 else 24 if tickets else 32)
        if merges:   # (trips to memory one after another; of long sequences they do not matter)
            assert -(-M * D // 256) * -(-live // 8) <= 4 or keys >= 1024
    assert not merges or -(-M * D // 256) <= 4


@pytest.mark.parametrize("room", [8192, 32768, 131072])
def test_room_hardly_counts(room):
    """The share of a short sequence that a workgroup has: not the 1,024 keys that a large cache's share is."""
    assert _plan(room, 4, 8, 4, 64, 700)[1] == 128
    assert 256 <= _plan(room, 13, 8, 4, 128, 1500)[1] <= 896
    assert 128 <= _plan(room, 1, 8, 4, 128, 1000)[1] <= 192


@pytest.mark.parametrize("B,T,H,G,D,most", [(1, 4, 8, 4, 128, 16), (1, 4, 8, 4, 64, 16), (1, 1, 8, 4, 64, 24), (1, 2, 8, 4, 128, 16)])
def test_few_heads_of_long_sequences(B, T, H, G, D, most):
    """64 splits took 1.2 to 2.6 times as long as 16."""
    splits, keys, merges = _plan(8192, B, H, G * T, D, 8000)
    assert splits <= most and splits * keys >= 8000 and merges == (T == 1)


@pytest.mark.gpu
@pytest.mark.parametrize("D,Hkv,G,T,L,lengths", [
    (64, 8, 4, 1, 8192, [700, 0, 1, 129]), (64, 1, 4, 1, 8192, [8192]), (64, 1, 4, 1, 4096, [3073, 3072, 3071]),
    (128, 8, 4, 4, 2304, [2000]), (128, 2, 4, 2, 8192, [4097, 130]), (64, 2, 4, 1, 70000, [69999, 500]), (128, 1, 1, 4, 2100, [2049]),
])
def test_attention_of_short_sequences_in_large_caches(D, Hkv, G, T, L, lengths):
    from test_decode_attention_splits_gpu import _reference

    dev, B = torch.device("cuda", 0), len(lengths)
    g = torch.Generator(device=dev).manual_seed(L + D)
    rand = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)
    q, k, v = rand(B, T, Hkv * G, D), rand(B, Hkv, L, D), rand(B, Hkv, L, D)
    for b, n in enumerate(lengths):   # keys past the end are never read
        k[b, :, n:] = float("nan")
        v[b, :, n:] = float("nan")
    n32 = torch.tensor(lengths, dtype=torch.int32, device=dev)
    ref = _reference(q, k, v, lengths, range(B))
    for tickets in (None, torch.zeros(B * Hkv, dtype=torch.int32, device=dev)):
        for _ in range(2):
            out = ops.decode_attention(q, k, v, n32, tickets=tickets).double().cpu()
            # probabilities and the result are rounded to bf16 (2^-9 each, relative); probabilities err independently
            err, rms = (out - ref).abs(), lambda x: x.pow(2).mean().sqrt().item()
            assert torch.isfinite(out).all() and rms(err) <= 2.0 ** -8 * rms(ref)
            assert (err <= 2.0 ** -9 * ref.abs() + 2.0 ** -8 * 4.5 * 0.25 + 1e-6).all()   # (values up to 4.5 or so)
        assert tickets is None or not tickets.any()
