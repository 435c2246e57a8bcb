"""The AdamW kernel at the edges of its blocks of 4,096 parameters, against the same step in float64; what lies behind the
last parameter stays."""
import pytest
import torch

from neuronx_distributed_llama3_2_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grad", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("out", [True, False])
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 1029, 4092, 4095, 4096, 4097, 8191, 3 * 4096 + 1026,
                               (1 << 21) - 3, (1 << 21) + 1029, (1 << 26) - 1025, (1 << 26) + 2051])   # (1, 2 and 4 vectors a thread)
def test_adamw_at_block_edges(n, out, grad):
    gen = torch.Generator(device="cuda").manual_seed(n)
    full = [torch.randn(n + 16, generator=gen, device="cuda") for _ in range(4)]
    full[2].square_()
    p, m, v, g = (t[:n] for t in full)
    g = g.to(grad)
    w = torch.full((n + 16,), 7.0, device="cuda", dtype=torch.bfloat16)
    start = [t.clone() for t in full]
    lr, b1, b2, eps, wd, step = 1e-3, 0.9, 0.95, 1e-8, 0.1, 3
    ops.adamw_flat_(p, g, m, v, w[:n] if out else None, lr, b1, b2, eps, wd, step, grad_scale_host=0.5)
    gd = g.double() * 0.5
    md = b1 * start[1][:n].double() + (1 - b1) * gd
    vd = b2 * start[2][:n].double() + (1 - b2) * gd * gd
    pd = start[0][:n].double() * (1 - lr * wd) - lr / (1 - b1 ** step) * md / ((vd / (1 - b2 ** step)).sqrt() + eps)
    # a handful of fp32 roundings (2^-24) of each term; the hyperparameters themselves are fp32: 8 of them
    near = lambda a, b, terms: ((a.double() - b).abs() <= 8 * 2.0 ** -23 * terms).all()
    assert near(m, md, start[1][:n].double().abs() + gd.abs())
    assert near(v, vd, vd.abs())
    assert near(p, pd, start[0][:n].double().abs() + (pd - start[0][:n].double()).abs() + 1e-2)   # (a step of many parameters may be large)
    if out:
        assert torch.equal(w[:n], p.bfloat16())
    assert (w[n if out else 0:] == 7).all()
    for t, s in zip(full[:3], start):
        assert torch.equal(t[n:], s[n:])
