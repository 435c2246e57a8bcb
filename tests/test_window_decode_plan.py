"""Which kernel takes a step of windowed attention, and in how many parts: on the matrix instructions unless the sizes are not theirs or few
pairs of a sequence and a key / value head have many query heads or few keys; no more parts than their merge pays for.  Both sides of
each line against float64."""
import pytest
import torch

from test_golitar_mechanisms import Attn
from test_window_decode_mfma_gpu import _exact

from neuronx_distributed_llama3_2_amd import ops


def _plan(B, sizes, seen, f32=False):
    return ops.hybrid_ext().attn_decode_plan(B, list(sizes), seen, f32)


@pytest.mark.parametrize("B,sizes,seen,mfma", [
    (16, (16, 4, 2, 64, 128), 1024, True), (1, (16, 4, 2, 64, 128), 1024, True), (16, (16, 4, 2, 64, 128), 33, True),
    (1, (4, 1, 1, 128, 64), 512, False), (1, (4, 1, 1, 128, 64), 513, True), (16, (4, 1, 1, 128, 64), 33, True),               # one map, few keys
    (16, (16, 1, 1, 64, 64), 512, False), (17, (16, 1, 1, 64, 64), 512, True),
    (8, (16, 1, 1, 64, 64), 1131, False), (8, (16, 1, 1, 64, 64), 1132, True), (1, (16, 1, 1, 64, 64), 25600, False), (12, (16, 1, 1, 64, 64), 1024, True),
    (2, (8, 1, 1, 64, 64), 1600, False), (2, (8, 1, 1, 64, 64), 1601, True), (4, (8, 1, 2, 64, 128), 1131, False), (4, (8, 1, 2, 64, 128), 1132, True),
    (40, (18, 1, 1, 64, 64), 1024, False), (40, (16, 4, 2, 48, 96), 1024, False), (40, (16, 4, 2, 64, 256), 1024, False)])
def test_kernel(B, sizes, seen, mfma):
    assert _plan(B, sizes, seen)[0] == mfma and not _plan(B, sizes, seen, True)[0]


@pytest.mark.parametrize("B,sizes,seen,splits", [
    (16, (16, 4, 2, 64, 128), 1024, 4), (1, (4, 1, 1, 128, 128), 1024, 8), (1, (4, 1, 1, 128, 128), 4096, 16), (1, (4, 1, 1, 128, 128), 16384, 37),
    (2, (8, 1, 1, 64, 64), 4096, 16), (2, (8, 1, 1, 64, 64), 16384, 24), (4, (16, 1, 1, 64, 64), 16384, 16), (64, (4, 4, 1, 64, 64), 16384, 1)])
def test_parts(B, sizes, seen, splits):
    mfma, share, n, tiles = _plan(B, sizes, seen)
    assert mfma and share == sizes[0] // sizes[1] and n == splits and 64 * n * tiles >= seen > 64 * (n - 1) * tiles


@pytest.mark.gpu
@pytest.mark.parametrize("B,sizes,window", [(8, (16, 1, 1, 64, 64), 1100), (8, (16, 1, 1, 64, 64), 1140), (1, (4, 1, 1, 128, 64), 3000),
                                            (4, (8, 1, 2, 64, 128), 1100), (4, (8, 1, 2, 64, 128), 1140), (2, (8, 1, 1, 128, 128), 1700)])
def test_at_the_lines(B, sizes, window):
    a = Attn(("cuda", torch.bfloat16, None), B, 1, *sizes, 16, window, 20.0, cap=window, seed=B)
    a.kc.normal_(generator=torch.Generator(device="cuda").manual_seed(1))
    a.vc.normal_(generator=torch.Generator(device="cuda").manual_seed(2))
    at = [window - 1, 3 * window // 2, 63, 64, window // 2, 0, 2 * window - 1, 127, 1]
    pos = torch.tensor([at[b % len(at)] % 4096 for b in range(B)], device="cuda")[:, None]
    buf = a.buf[:, 0].contiguous()
    prep = (a.bias.cuda(), a.qn.cuda(), a.kn.cuda(), 1e-5, a.cos.cuda(), a.sin.cuda(), pos)
    row, kw, vw = buf.clone(), a.kc.clone(), a.vc.clone()
    ops.attn_prep_(row, B, 1, a.sz, *prep, None, a.slots, kw, vw)
    want = _exact(a, row, kw, vw, pos)
    got = ops.attn_decode(buf, a.sz, a.rule, *prep, a.slots, a.kc, a.vc, a.tickets).double()
    assert int(a.tickets.abs().sum()) == 0 and torch.equal(a.vc, vw)
    # results are rounded to bf16, half an ulp 2^-8 at the most; queries and the new key may be rounded the other way
    assert ((got - want).norm(dim=1) <= 2 ** -8 * want.norm(dim=1)).all()
