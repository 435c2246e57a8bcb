"""The chunked delta rule's scan in two launches (few blocks of columns) gives the bits of the one launch that a larger batch takes, and the oracle's
numbers: ragged lengths, head sizes that fill no block, a state that goes on, keys of more than 128,
outputs normed where they are formed, in both activation types."""
import pytest
import torch

from test_golitar_mechanisms import delta_case, delta_oracle, rel_err, run_delta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 5e-5), (torch.bfloat16, 2e-2)], ids=["f32", "bf16"])   # (as in test_golitar_mechanisms)
@pytest.mark.parametrize("H,G,D,V,T", [(3, 3, 16, 24, 300), (16, 8, 128, 128, 769), (2, 1, 70, 33, 1000), (9, 9, 144, 16, 130), (4, 2, 256, 40, 250),
                                       (16, 8, 32, 68, 2100), (16, 16, 128, 128, 2049)])   # (16 heads: the outputs' launch norms them)
def test_two_launches(H, G, D, V, T, dtype, tol):
    from neuronx_distributed_llama3_2_amd import ops

    where, taps = ("cuda", dtype, tol), 4
    n = -(-257 // (H * -(-V // 16))) + 1          # sequences of the batch that takes one launch
    lens = [T, T - 67] + [1] * (n - 2)
    case = delta_case(where, n, T, H, G, D, V, taps)
    sz, proj, proj_o = case[:3]

    def run(rows, pos0, state, ring):
        t = torch.tensor
        B = len(rows)
        print(H, G, D, V, T, B, dtype, flush=True)
        return ops.delta_rule(proj[rows].reshape(B * T, -1).contiguous(), B, T, sz, *(v.cuda() for v in case[3:]), 1e-5,
                              t([pos0] * B, device="cuda"), t([lens[r] for r in rows], dtype=torch.int32, device="cuda"), None, state, ring).view(B, T, H, V)

    def fresh(B):
        g = torch.Generator().manual_seed(5)
        return (torch.randn((1, H, V, sz.padded_dim), generator=g).expand(B, -1, -1, -1).contiguous().cuda(),
                torch.zeros((B, taps, sz.channels), dtype=dtype, device="cuda"))

    for pos0 in (0, 64):                           # a prompt, and one that goes on from a state
        s_all, r_all = fresh(n)
        y_all = run(list(range(n)), pos0, s_all, r_all)
        for r in (0, 1):
            s, ring = fresh(1)
            y = run([r], pos0, s, ring)
            assert not y[0, lens[r]:].any() and not y_all[r, lens[r]:].any()
            assert torch.equal(y[0, :lens[r]], y_all[r, :lens[r]]) and torch.equal(s[0], s_all[r]) and torch.equal(ring[0], r_all[r])
    for pos0 in (0, 64):                           # (at 64 with a state, and no inputs before it)
        st, ring = fresh(1)
        before = st[0, :, :, :D].transpose(1, 2).double().cpu() if pos0 else None
        got = run([1], pos0, st, ring)
        assert rel_err(got[0, :lens[1]].reshape(lens[1], -1), delta_oracle(sz, proj_o[1, :lens[1]], *case[3:], 1e-5, before)) < tol


def test_without_room_for_the_states():
    """Room for the one launch's operands and not for the states beside them: the same bits, and the scratch is given back."""
    from neuronx_distributed_llama3_2_amd import ops

    H, D, V, T, taps = 16, 128, 128, 8192, 4                     # operands of the chunks 169 MB, states and U 201 MB
    case = delta_case(("cuda", torch.bfloat16, 0), 1, T, H, H, D, V, taps)
    sz, proj = case[0], case[1][0].contiguous()
    rest = [v.cuda() for v in case[3:]]

    def run():
        state = torch.zeros((1, H, V, sz.padded_dim), device="cuda")
        ring = torch.zeros((1, taps, sz.channels), dtype=torch.bfloat16, device="cuda")
        y = ops.delta_rule(proj, 1, T, sz, *rest, 1e-5, torch.zeros(1, dtype=torch.long, device="cuda"), None, None, state, ring)
        return y.cpu(), state.cpu(), ring.cpu()

    want = run()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # what the call has beside them: q, k of all heads, v and o, gates in fp32, y, and blocks of 2 MB or 20 MB that the allocator rounds to
    need = 4 * (4 * T * H * D + 2 * T * H) + 2 * T * H * V + 4 * 2 ** 20 * 16
    operands = T // 64 * H * 64 * (D + V + 64 + 2) * 4
    reserved, total = torch.cuda.memory_reserved(), torch.cuda.get_device_properties(0).total_memory
    held = []
    try:
        torch.cuda.set_per_process_memory_fraction(reserved / total)
        for size in (2 ** e for e in range(30, 20, -1)):         # (room that others have left within their blocks)
            try:
                while True:
                    held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            except torch.cuda.OutOfMemoryError:
                pass
        torch.cuda.set_per_process_memory_fraction((reserved + need + operands + 64 * 2 ** 20) / total)
        before = torch.cuda.memory_stats()["num_ooms"]
        got = run()
        assert torch.cuda.memory_stats()["num_ooms"] > before    # (there was no room)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
