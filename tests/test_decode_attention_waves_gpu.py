"""Decode attention in parts of 8 waves and its lines to those of 4: whole heads, several parts a head, parts' ends, empty
sequences, keys past the end, several new tokens.  Against float64."""
import pytest
import torch

from test_decode_attention_splits_gpu import _reference

from neuronx_distributed_llama3_2_amd import ops


@pytest.mark.parametrize("room,B,Hkv,M,D,keys", [
    (640, 4, 8, 4, 64, 640), (641, 4, 8, 4, 64, 256), (2304, 32, 8, 4, 64, 2304), (2560, 28, 8, 4, 64, 2560),      # whole heads, 8 parts
    (2561, 32, 8, 4, 64, 1024), (1281, 20, 8, 4, 64, 448), (1280, 20, 8, 4, 64, 1280), (2304, 16, 8, 4, 64, 1152),
    (2304, 12, 8, 4, 64, 448), (1280, 1, 8, 4, 64, 128), (1281, 1, 8, 4, 64, 256), (4608, 8, 8, 4, 64, 1152), (4609, 8, 8, 4, 64, 640),
    (1756, 13, 8, 4, 128, 640), (640, 20, 8, 4, 128, 320), (641, 24, 8, 4, 128, 256), (1, 32, 8, 16, 128, 256), (2304, 1, 8, 4, 128, 192),
])
def test_keys_of_a_part(room, B, Hkv, M, D, keys):
    assert ops.ext().decode_attn_plan(room, B, Hkv, M, D, room, True)[1] == keys


@pytest.mark.gpu
@pytest.mark.parametrize("D,B,Hkv,G,T,L", [(64, 32, 8, 4, 1, 300), (64, 4, 8, 4, 1, 640), (64, 5, 8, 4, 2, 1281), (64, 32, 8, 2, 1, 1000), (64, 16, 8, 4, 4, 900),
                                           (128, 13, 8, 4, 1, 640), (128, 1, 8, 4, 1, 1500), (128, 3, 8, 1, 4, 700), (128, 32, 8, 4, 1, 300), (128, 24, 8, 4, 1, 641)])
def test_attention(D, B, Hkv, G, T, L):
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(L + D)
    rand = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)  # noqa: E731
    lengths = [n for n in (L, 0, 1, 31, 32, 33, 255, 256, 257, L - 1, 511, 513, L // 2) if n <= L]
    lengths = [lengths[i % len(lengths)] for i in range(B)]
    lengths = [n if n == 0 or n >= T else T for n in lengths]
    q, k, v = rand(B, T, Hkv * G, D), rand(B, Hkv, L, D), rand(B, Hkv, L, D)
    for b, n in enumerate(lengths):   # keys past the end are never read
        k[b, :, n:] = float("nan")
        v[b, :, n:] = float("nan")
    n32 = torch.tensor(lengths, dtype=torch.int32, device=dev)
    ref = _reference(q, k, v, lengths, range(B))
    tickets = torch.zeros(B * Hkv, dtype=torch.int32, device=dev)
    for _ in range(2):
        out = ops.decode_attention(q, k, v, n32, tickets=tickets).double().cpu()
        # probabilities and the result are rounded to bf16 (2^-9 each, relative); probabilities err independently
        err, rms = (out - ref).abs(), lambda x: x.pow(2).mean().sqrt().item()  # noqa: E731
        assert torch.isfinite(out).all() and rms(err) <= 2.0 ** -8 * rms(ref)
        assert (err <= 2.0 ** -9 * ref.abs() + 2.0 ** -8 * 4.5 * 0.25 + 1e-6).all()   # (values up to 4.5 or so)
    assert not tickets.any()
