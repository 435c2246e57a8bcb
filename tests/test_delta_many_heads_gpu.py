"""The delta rule's launches whose work is shared by heads and columns: several parts of the heads, the last one short or empty of
values, keys of more than 128 (fewer waves).  Against the oracle in float64."""
import pytest
import torch

from test_golitar_mechanisms import delta_case, delta_oracle, rel_err, run_delta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", [("cuda", torch.float32, 5e-5), ("cuda", torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("H,G,D,V,taps", [(16, 16, 16, 24, 4), (10, 5, 33, 20, 3), (40, 20, 8, 130, 4), (9, 9, 144, 16, 5)])
def test_delta_rule(where, H, G, D, V, taps):
    B, T, lens = 2, 75, [75, 41]
    case = delta_case(where, B, T, H, G, D, V, taps)
    sz, proj, proj_o = case[:3]
    want = [delta_oracle(sz, proj_o[b, :lens[b]], *case[3:], 1e-5) for b in range(B)]
    for cuts, chunk_from in (([75], 32), ([75], 1000), ([33, 2, 40], 2)):
        state = torch.zeros((2, H, V, sz.padded_dim), device="cuda")
        ring = torch.zeros((2, taps, sz.channels), dtype=where[1], device="cuda")
        got = run_delta(where, case, cuts, lens, torch.tensor([1, 0], dtype=torch.int32), state, ring, chunk_from)
        for b in range(B):
            assert rel_err(got[b, :lens[b]], want[b]) < where[2], (cuts, chunk_from, b)
