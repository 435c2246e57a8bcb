"""Decode attention on the matrix instructions against the one-wave-a-query kernel on the same cache: few and many keys around its
chunks and parts, a wrapped ring, queries that fill the 16 rows or hardly any, stale NaNs in the new key's place."""
import pytest
import torch

from test_golitar_mechanisms import Attn

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,window,softcap", [(1, 1, 20.0), (3, 33, 0.0), (2, 130, 20.0), (5, 1000, 20.0), (40, 300, 0.0)])
@pytest.mark.parametrize("H,G,R,D,V", [(16, 4, 2, 64, 128), (8, 1, 2, 64, 64), (16, 1, 1, 128, 128), (4, 4, 1, 128, 64), (6, 2, 2, 128, 128),
                                       (5, 1, 1, 64, 64), (18, 1, 1, 64, 64)])   # the last: more than 16 rows, the kernel of any size
def test_against_a_wave_a_query(B, window, softcap, H, G, R, D, V):
    T = 2 * window + 40
    where = ("cuda", torch.bfloat16, None)
    a = Attn(where, B, T, H, G, R, D, V, 16, window, softcap, cap=window + 15, seed=B)
    a.kc.normal_(generator=torch.Generator(device="cuda").manual_seed(1))
    a.vc.normal_(generator=torch.Generator(device="cuda").manual_seed(2))
    at = [0, 1, 30, 31, 32, 63, 64, 127, 128, 129, window - 1, window, window + 14, window + 15, T - 1]
    pos = torch.tensor([min(at[(B + 4 * i) % len(at)], T - 1) for i in range(B)], device="cuda")[:, None]
    buf = a.buf[:, T - 1].contiguous()
    prep = (a.bias.cuda(), a.qn.cuda(), a.kn.cuda(), 1e-5, a.cos.cuda(), a.sin.cuda(), pos)
    row, kw, vw = buf.clone(), a.kc.clone(), a.vc.clone()
    ops.attn_prep_(row, B, 1, a.sz, *prep, None, a.slots, kw, vw)
    want = ops.window_attention(row, B, 1, a.sz, a.rule, pos, None, a.slots, kw, vw, False, False)
    e = pos[:, 0] % a.cap
    a.kc.view(B + 1, G, R, a.cap, D)[a.slots.long(), :, :, e] = float("nan")
    a.vc[a.slots.long(), :, e] = float("nan")
    got = ops.attn_decode(buf, a.sz, a.rule, *prep, a.slots, a.kc, a.vc, a.tickets)
    assert int(a.tickets.abs().sum()) == 0 and torch.equal(a.vc, vw)
    # the key: the same sums in another order, a rounding to bf16
    assert (a.kc.float() - kw.float()).abs().max() <= 2 ** -7 * kw.float().abs().max()
    # one rounding to bf16 of the results (2^-8 relative) and, where a query or the new key was rounded the other way, that score
    err = (got.double() - want.double()).norm() / want.double().norm()
    assert err < 2 ** -7, err


def _exact(a, row, kc, vc, pos):
    """float64, from prepared queries (in row) and a cache that has the new key"""
    sz, rule, out = a.sz, a.rule, []
    for b in range(a.B):
        ps, slot = int(pos[b]), int(a.slots[b])
        at = torch.arange(max(0, ps - a.window + 1, ps - a.cap + 1), ps + 1, device=row.device) % a.cap
        q = row[b, :sz.q_columns].double().view(sz.kv_heads, -1, sz.maps, sz.dim)
        k = kc[slot].double().view(sz.kv_heads, sz.maps, a.cap, sz.dim)[:, :, at]
        s = (q[:, :, :, None] * k[:, None]).sum(-1) * rule.scale
        s = rule.softcap * torch.tanh(s / rule.softcap) if rule.softcap else s
        o = (s.softmax(-1)[..., None] * vc[slot].double()[:, None, None, at]).sum(-2)
        if sz.maps == 2:
            o = o[:, :, 0] - rule.lam * o[:, :, 1]
            o = o / (o.square().mean(-1, keepdim=True) + rule.eps).sqrt()
        out.append((o * rule.out_scale).reshape(-1))
    return torch.stack(out)


@pytest.mark.parametrize("what", ["key", "value", "new value"])
@pytest.mark.parametrize("B,window", [(2, 33), (3, 300), (40, 130)])
@pytest.mark.parametrize("H,G,R,D,V", [(16, 4, 2, 64, 128), (8, 1, 2, 128, 64), (16, 1, 1, 128, 128), (40, 8, 1, 64, 64)])
def test_infinities(B, window, H, G, R, D, V, what):
    """An infinite key leaves the scores of the other map alone and is bounded by the cap in its own; an infinite value gives
    infinities in its column and nowhere else (with two maps, whose difference is normalised, NaNs in its heads)."""
    if R == 1 and B * G < 16 and window <= 512 and what == "new value":
        pytest.skip("not on the matrix instructions")
    T = window + 60
    a = Attn(("cuda", torch.bfloat16, None), B, T, H, G, R, D, V, 16, window, 20.0, cap=window + 15, seed=B)
    a.kc.normal_(generator=torch.Generator(device="cuda").manual_seed(1))
    a.vc.normal_(generator=torch.Generator(device="cuda").manual_seed(2))
    pos = torch.tensor([window + 3 + 7 * (b % 5) for b in range(B)], device="cuda")[:, None]
    slots = a.slots.long()
    for b in range(B):   # some visible keys of some key / value heads
        for i, (back, sign) in enumerate([(1, 1), (window // 2, -1), (window - 1, 1)]):
            e, g, inf = int(pos[b] - back) % a.cap, (b + i) % G, sign * float("inf")
            if what == "key":
                a.kc[slots[b], g * R + (b + i) % R, e, 3 * i + 1] = inf
            elif what == "value":
                a.vc[slots[b], g, e, 5 * i % 10 + b % 2] = inf
    buf = a.buf[:, T - 1].contiguous()
    if what == "new value":
        buf[:, (H + G) * R * D + 7] = float("inf")
    prep = (a.bias.cuda(), a.qn.cuda(), a.kn.cuda(), 1e-5, a.cos.cuda(), a.sin.cuda(), pos)
    row, kw, vw = buf.clone(), a.kc.clone(), a.vc.clone()
    ops.attn_prep_(row, B, 1, a.sz, *prep, None, a.slots, kw, vw)
    want = _exact(a, row, kw, vw, pos)
    got = ops.attn_decode(buf, a.sz, a.rule, *prep, a.slots, a.kc, a.vc, a.tickets).double()
    finite = torch.isfinite(want)
    assert finite.all() if what == "key" else not finite.all()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
    # one rounding to bf16 of the results, and queries that were rounded the other way
    if finite.any():
        err = (got[finite] - want[finite]).norm() / want[finite].norm()
        assert err < 2 ** -7, err
