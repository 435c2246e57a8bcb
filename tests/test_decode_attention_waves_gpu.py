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


@pytest.mark.parametrize("room,B,M,splits,keys", [
    (1024, 5, 4, 6, 192), (1024, 5, 8, 6, 192), (1536, 5, 4, 6, 256), (1280, 8, 4, 4, 320), (1024, 10, 4, 3, 384), (768, 13, 4, 2, 384), (512, 20, 4, 1, 512),
    (640, 13, 4, 3, 256), (1756, 13, 4, 3, 640), (2304, 5, 4, 8, 320),                                  # the last part half empty; longer parts
    (1024, 5, 16, 6, 192), (1280, 8, 16, 4, 320), (1280, 10, 12, 3, 448), (1536, 13, 16, 2, 768),       # merged by a launch of its own
    (640, 7, 16, 5, 128), (768, 6, 16, 6, 128), (384, 8, 12, 3, 128), (512, 8, 16, 4, 128), (640, 8, 16, 3, 256),
    (1280, 20, 16, 2, 640), (1279, 20, 16, 3, 448)])
def test_no_second_round(room, B, M, splits, keys):
    """8 heads of 128: parts that all have keys are no more than a round of workgroups; where a launch merges them no parts are."""
    assert ops.ext().decode_attn_plan(room, B, 8, M, 128, room, True)[:2] == (splits, keys)


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,L", [(5, 4, 1024), (7, 4, 640), (8, 3, 384), (13, 4, 768), (20, 1, 512), (10, 3, 1280)])
def test_attention_in_one_round(B, T, L):
    g = torch.Generator(device="cuda").manual_seed(L + B)
    q, k, v = (torch.randn(s, generator=g, device="cuda").bfloat16() for s in ((B, T, 32, 128), (B, 8, L, 128), (B, 8, L, 128)))
    lengths = [max(n, T) for n in (L, 1, 255, 257, L - 1, L // 2, 129, 321, 0)]
    lengths = [min(lengths[i % len(lengths)], L) for i in range(B)]
    for b, n in enumerate(lengths):   # keys past the end are never read
        k[b, :, n:] = float("nan")
        v[b, :, n:] = float("nan")
    tickets = torch.zeros(B * 8, dtype=torch.int32, device="cuda")
    out = ops.decode_attention(q, k, v, torch.tensor(lengths, dtype=torch.int32, device="cuda"), tickets=tickets).double().cpu()
    ref, size = (_reference(q, k, x, lengths, range(B)) for x in (v, v.abs()))
    # half an ulp of bf16 (8 significant bits) of the result and of each probability: 2^-8 of |result| and of the sum of p |v|; fp32 sums
    assert ((out - ref).abs() <= 2.0 ** -8 * (ref.abs() + size) + 2.0 ** -16 * size).all() and not tickets.any()
