"""The target's term of the loss gradient at the edges of a thread's chunks, for every width that a row's registers are laid out for."""
import pytest
import torch

from trainium_frontier_them_bones_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [0.0, 15.0])
@pytest.mark.parametrize("V", [8, 1024, 2048, 2056, 8192, 8200, 16384, 32760, 32768, 50304, 65536])
def test_target_column(V, cap):
    dev = torch.device("cuda:0")
    t = [0, 1, 7, 8 % V, V // 2, V - 8, V - 7, V - 1, -1, -8, V, V + 7, 2**32 + 3, -2**32 + 3, 2**62]
    g = torch.Generator().manual_seed(V)
    x = (2 * torch.randn(len(t), V, generator=g)).bfloat16()
    tg = torch.tensor(t)
    w = 0.5 + torch.rand(len(t), generator=g)
    live = (tg >= 0) & (tg < V)
    xd = x.double()
    s = cap * torch.tanh(xd / cap) if cap else xd
    p = torch.softmax(s, 1)
    p[live.nonzero()[:, 0], tg[live]] -= 1.0
    ref = (w.double() * live)[:, None] * p * ((1 - torch.tanh(xd / cap) ** 2) if cap else 1.0)
    y = x.to(dev)
    rows, lse = ops.loss_fwd_bwd(y, tg.to(dev), w.to(dev), cap)
    two = ops.loss_bwd(x.to(dev), tg.to(dev), lse, w.to(dev), cap)
    assert torch.equal(y, two)
    # one rounding to bf16 (2^-9 of the value) and fp32 before it: an exponential of an argument below 32 is off by 32 * 2^-23 of a
    # probability of at most one, the tanh's factor by a few 2^-23
    err = (y.cpu().double() - ref).abs()
    assert bool((err <= 2.0**-8 * ref.abs() + 1e-5).all()), float((err - 2.0**-8 * ref.abs()).max())
    assert not y[~live.to(dev)].any() and not rows[~live.to(dev)].any()
    if V > 8:  # int32 targets take the same columns
        z = x.to(dev)
        ops.loss_fwd_bwd(z, tg.clamp(-1, V).int().to(dev), w.to(dev), cap)
        assert torch.equal(y, z)


@pytest.mark.parametrize("cap", [0.0, 15.0])
@pytest.mark.parametrize("V,n", [(24, 8188), (24, 8189), (2048, 8195), (2056, 2047), (2056, 2048), (8200, 2049), (16392, 2050), (32776, 2048)])
def test_long_launches_take_the_same_bits(V, n, cap):
    # a launch of 2048 blocks and more may go through its values in another order than one of a few rows: no bit depends on it
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(V + n)
    x = (3 * torch.randn(n, V, generator=g, device=dev)).bfloat16()
    tg = torch.randint(-2, V + 2, (n,), generator=g, device=dev)
    w = 0.5 + torch.rand(n, generator=g, device=dev)
    for t in (tg, tg.int()):
        y = x.clone()
        rows, lse = ops.loss_fwd_bwd(y, t, w, cap)
        two = ops.loss_bwd(x, t, lse, w, cap)
        assert torch.equal(y, two)
        for a in range(0, n, 1000):
            b = min(a + 1000, n)
            z = x[a:b].clone()
            r, l = ops.loss_fwd_bwd(z, t[a:b].contiguous(), w[a:b].contiguous(), cap)
            assert torch.equal(z, y[a:b]) and torch.equal(r, rows[a:b]) and torch.equal(l, lse[a:b])
            assert torch.equal(ops.loss_bwd(x[a:b].contiguous(), t[a:b].contiguous(), l, w[a:b].contiguous(), cap), z)
