"""Rotation and cache write in one launch against the two launches: every head size, odd rows, entries before and past the cache's
ends, other cache rows; layouts that it does not take go to the two."""
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
