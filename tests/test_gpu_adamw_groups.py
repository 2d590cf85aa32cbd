"""AdamW at the edges of a thread's group of four and of a workgroup's 256 elements: every element once, none behind the last."""
import pytest
import torch

from trainium_frontier_them_bones_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 5, 252, 255, 256, 257, 260, 511, 512, 1026, 65536, 65793])
@pytest.mark.parametrize("g_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("copy", [True, False])
def test_every_element_once(n, g_dtype, copy):
    from oracle import optim as O
    dev, pad = torch.device("cuda:0"), 16
    gen = torch.Generator().manual_seed(n)
    p, m, v = torch.randn(n + pad, generator=gen), 0.1 * torch.randn(n + pad, generator=gen), torch.rand(n + pad, generator=gen)
    g = torch.randn(n + pad, generator=gen).to(g_dtype)
    pd, md, vd, gd = (t.to(dev) for t in (p, m, v, g))
    p16 = torch.full((n + pad,), 7.0, dtype=torch.bfloat16, device=dev)
    ops.adamw_(pd[:n], gd[:n], md[:n], vd[:n], 3, 3e-4, 0.9, 0.95, 1e-8, 0.1, p16[:n] if copy else None)
    want = [t[:n].clone() for t in (p, m, v)]
    O.adamw_step(want[0], g[:n], want[1], want[2], 3, 3e-4, 0.9, 0.95, 1e-8, 0.1)
    for got, was, w in zip((pd, md, vd), (p, m, v), want):
        # a few roundings of 2^-24 of values below 8
        assert torch.equal(got[n:].cpu(), was[n:]) and (got[:n].cpu() - w).abs().max().item() < 2e-6
        assert not torch.equal(got[:n].cpu(), was[:n])
    assert bool((p16[n:] == 7.0).all()) and torch.equal(p16[:n], pd[:n].bfloat16() if copy else torch.full_like(p16[:n], 7.0))
