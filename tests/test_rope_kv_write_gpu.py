"""Rotation and cache write in one launch against the two launches: every head size, odd rows, entries before and past the cache's
ends, other cache rows, caches that are not aligned (the two).  Caches that neither takes are refused with the queries as they were."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B,T,nq,nkv,idx,view", [(1, 1, 1, 1, False, False), (3, 37, 4, 2, True, False), (2, 129, 8, 1, False, False), (2, 33, 0, 3, True, False),
                                                 (3, 20, 4, 2, True, True)])
def test_against_two_launches(B, T, nq, nkv, D, idx, view):
    g = torch.Generator(device="cuda").manual_seed(B * T + D)
    Lmax, W = 64, (nq + 2 * nkv) * D
    qkv = torch.randn(B, T, W, generator=g, device="cuda").bfloat16()
    pos0 = torch.tensor([5, -3, 40][:B], device="cuda", dtype=torch.int32)     # before the cache's first entry, past its last
    pos = (torch.arange(T, device="cuda")[None] + torch.tensor([7, 0, 90][:B], device="cuda")[:, None]).reshape(-1)
    ang = torch.rand(300, D // 2, generator=g, device="cuda") * 6
    cos, sin = ang.cos(), ang.sin()
    ci = torch.randperm(B + 1, generator=g, device="cuda")[:B].to(torch.int32) if idx else None
    shape = (2, B + 1, nkv, 2 * Lmax, D)
    a, b = (torch.full(shape, 7.0, device="cuda").bfloat16()[:, :, :, :Lmax] if view else torch.full(shape[:3] + (Lmax, D), 7.0, device="cuda").bfloat16()
            for _ in range(2))
    want = qkv.clone()
    ops.rope_inplace_(want.view(B * T, W), 0, nq + nkv, D, cos, sin, pos)
    h = want.view(B, T, nq + 2 * nkv, D)
    if view:   # (caches that are not contiguous: neither takes them)
        for f in (lambda: ops.kv_cache_write(h[:, :, nq:nq + nkv], h[:, :, nq + nkv:], a[0], a[1], pos0, ci),
                  lambda: ops.rope_kv_write_(qkv, nq, nkv, cos, sin, pos, b[0], b[1], pos0, ci)):
            with pytest.raises(RuntimeError):
                f()
        return
    ops.kv_cache_write(h[:, :, nq:nq + nkv], h[:, :, nq + nkv:], a[0], a[1], pos0, ci)
    ops.rope_kv_write_(qkv, nq, nkv, cos, sin, pos, b[0], b[1], pos0, ci)
    assert torch.equal(qkv, want) and torch.equal(a, b)


@pytest.mark.parametrize("what", ["view", "heads", "slots", "type"])
def test_refused_before_the_rotation(what):
    B, T, nq, nkv, D, L = 2, 5, 4, 2, 64, 16
    qkv = torch.randn(B, T, (nq + 2 * nkv) * D, device="cuda").bfloat16()
    cos, sin = (torch.randn(64, D // 2, device="cuda") for _ in range(2))
    pos, pos0 = torch.arange(T, device="cuda").repeat(B), torch.zeros(B, dtype=torch.int32, device="cuda")
    kc, vc = (torch.zeros(B, nkv, L, D, device="cuda").bfloat16() for _ in range(2))
    bad = {"view": (kc[:, :, :8], vc[:, :, :8]), "heads": (kc[:, :1].contiguous(), vc[:, :1].contiguous()), "slots": (kc[:1], vc[:1]),
           "type": (kc, vc.float())}[what]
    kept = qkv.clone()
    with pytest.raises(RuntimeError):
        ops.rope_kv_write_(qkv, nq, nkv, cos, sin, pos, *bad, pos0)
    assert torch.equal(qkv, kept)


def test_caches_of_any_alignment():
    B, T, nq, nkv, D, L = 2, 5, 4, 2, 64, 16
    qkv = torch.randn(B, T, (nq + 2 * nkv) * D, device="cuda").bfloat16()
    cos, sin = (torch.randn(64, D // 2, device="cuda") for _ in range(2))
    pos, pos0 = torch.arange(T, device="cuda").repeat(B), torch.tensor([3, 0], dtype=torch.int32, device="cuda")
    n = B * nkv * L * D
    caches = [[torch.zeros(n + 2, device="cuda").bfloat16()[at:at + n].view(B, nkv, L, D) for _ in range(2)] for at in (0, 2)]
    rows = [qkv.clone() for _ in caches]
    for q, (kc, vc) in zip(rows, caches):
        ops.rope_kv_write_(q, nq, nkv, cos, sin, pos, kc, vc, pos0)
    assert torch.equal(rows[0], rows[1]) and all(torch.equal(a, b) for a, b in zip(*caches)) and caches[0][0].any()
