"""Decode attention whose key splits are merged by the last of them to finish, against attention in float64: sequences of
every length around the splits' and chunks' edges (none and one key, a full cache), one and several new tokens, strided
queries and caches, more splits than are merged at once; counters stay zeroed and replays of a graph repeat the result."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu


def _reference(q, k, v, n, idx):
    B, T, Hq, D = q.shape
    G = Hq // k.shape[1]
    out = torch.zeros(B, T, Hq, D, dtype=torch.float64)
    q, k, v = q.double().cpu(), k.double().cpu(), v.double().cpu()
    for b in range(B):
        for t in range(T):
            m = n[b] - (T - 1 - t)
            if m <= 0:
                continue
            for h in range(Hq):
                p = torch.softmax(k[idx[b], h // G, :m] @ q[b, t, h] * D ** -0.5, 0)
                out[b, t, h] = p @ v[idx[b], h // G, :m]
    return out


@pytest.mark.parametrize("D,Hkv,G,T,L,lengths", [
    (64, 8, 4, 1, 700, [700, 0, 1, 127, 128, 129]),
    (64, 2, 4, 1, 2304, [2304, 2048, 1025, 33]),          # 18 splits: more than the 8 in flight
    (64, 1, 4, 4, 1000, [1000, 3, 257]),                  # 16 query rows, a row without keys
    (128, 8, 4, 1, 1756, [1500, 750, 1, 0, 512, 513]),
    (128, 1, 1, 2, 300, [300, 2, 96, 97, 129]),
    (128, 2, 8, 2, 1100, [1100, 640]),                    # 16 query rows
    (64, 8, 2, 1, 100, [100, 64]),                        # one split
])
def test_matches_reference(D, Hkv, G, T, L, lengths):
    dev, B = torch.device("cuda", 0), len(lengths)
    g = torch.Generator(device=dev).manual_seed(L + D)
    rand = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)
    q = rand(B, T, Hkv * G + 2 * Hkv, D)[:, :, :Hkv * G]           # heads of a joint projection
    k, v = rand(B + 1, Hkv, L, D), rand(B + 1, Hkv, L, D)
    idx = [(b + 1) % (B + 1) for b in range(B)]
    n32, i32 = (torch.tensor(x, dtype=torch.int32, device=dev) for x in (lengths, idx))
    tickets = torch.zeros(B * Hkv, dtype=torch.int32, device=dev)
    ref = _reference(q, k, v, lengths, idx)
    run = lambda t: ops.decode_attention(q, k, v, n32, i32, tickets=t)
    out = run(tickets)
    # probabilities and the result are rounded to bf16 (2^-9 each, relative); probabilities err independently
    err = (out.double().cpu() - ref).abs()
    bound = 2.0 ** -9 * ref.abs() + 2.0 ** -8 * v.float().abs().max().item() * 0.25 + 1e-6
    assert torch.isfinite(out.float()).all() and (err <= bound).all(), (err - bound).max()
    rms = lambda x: x.pow(2).mean().sqrt().item()
    assert rms(err) <= 2.0 ** -8 * rms(ref)
    assert rms((run(None).double().cpu() - ref)) <= 2.0 ** -8 * rms(ref)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        again = run(tickets)
    for _ in range(4):
        again.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(again, out) and not tickets.any()


def test_counters_are_checked():
    dev = torch.device("cuda", 0)
    q, k = torch.zeros(2, 1, 8, 64, device=dev, dtype=torch.bfloat16), torch.zeros(2, 2, 64, 64, device=dev, dtype=torch.bfloat16)
    n = torch.ones(2, dtype=torch.int32, device=dev)
    for bad in (torch.zeros(3, dtype=torch.int32, device=dev), torch.zeros(4, dtype=torch.int64, device=dev)):
        with pytest.raises(RuntimeError):
            ops.decode_attention(q, k, k, n, tickets=bad)
