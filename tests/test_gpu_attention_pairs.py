"""dK and dV by pairs of wavefronts, and dQ, over the forms a call may have. At D = 64, and for dQ at D = 128, a launch of many blocks runs one
wavefront to 32 tokens, and a launch of few in pairs has its bits. dK and dV of D = 128 always run in pairs: there the launches say that the
grid does not matter, and the comparison with fp32 is what holds the values."""
import pytest
import torch

from trainium_frontier_them_bones_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _grads(B, T, H, D, band, rope, qkv, do):
    q, k, v = (t.view(B, T, H, D) for t in qkv.split(H * D, dim=-1))
    kw = {"band": band} if band else {}
    o, lse = ops.attn_fwd(q, k, v, D ** -0.5, layout="bthd", **kw)
    out = torch.full_like(qkv, float("nan"))
    dq, dk, dv = (t.view(B, T, H, D) for t in out.split(H * D, dim=-1))
    ops.attn_bwd(q, k, v, o, do, lse, D ** -0.5, "bthd", dq, dk, dv, "bthd", rope=rope, **kw)
    return out


# two blocks (the fewest that D = 64 has in pairs) and one (which it has not, nor has a band of one), odd and even numbers of blocks, bands,
# and the most blocks: about one for each CU of short sequences and two of long ones (31 heads: two blocks a workgroup), less for dQ. pairs: what runs in pairs at D = 64 and at
# D = 128 (1 = dQ, 2 = dK and dV); of the other launch nothing may at D = 64.
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T,H,band,rope,pairs", [
    (128, 3, 0, True, (1, 3)), (256, 2, 0, True, (3, 3)), (256, 2, 1, False, (1, 3)), (384, 1, 0, False, (3, 3)), (640, 2, 2, True, (3, 3)),
    (1024, 3, 0, True, (3, 3)), (1152, 1, 3, False, (3, 3)), (1536, 2, 0, True, (3, 3)), (2048, 1, 1, False, (1, 3)), (512, 64, 0, False, (2, 2)),
    (2048, 19, 0, True, (3, 3)), (2048, 24, 0, False, (3, 2)), (2048, 31, 0, True, (2, 2)), (2048, 33, 0, True, (2, 2)), (1024, 32, 2, False, (2, 2))])
def test_key_and_value_gradients_in_pairs(T, H, band, rope, pairs, D):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(T + H + band)
    many = -(-4 * 256 * 128 // (T * H))
    routes = [sum(w for w in (1, 2) if _lib.lib().tfb_attn_bwd_pairs_applies(w, n, H, T, D, band) == 0) for n in (1, many)]
    assert routes == [pairs[D // 128], 0 if D == 64 else 2]
    qkv = torch.randn(1, T, 3 * H * D, generator=g, device=dev).bfloat16()
    do = torch.randn(1, T, H, D, generator=g, device=dev).bfloat16()
    tables = None
    if rope and D == 64:
        from oracle import attention as O
        tables = tuple(t.to(dev) for t in O.rope_tables(T, D))
    few = _grads(1, T, H, D, band, tables, qkv, do)
    lot = _grads(many, T, H, D, band, tables, qkv.expand(many, -1, -1).contiguous(), do.expand(many, -1, -1, -1).contiguous())
    assert torch.equal(few[0], lot[-1]) and torch.equal(lot[0], lot[-1])
    q, k, v = (t.view(1, T, H, D).permute(0, 2, 1, 3).float().requires_grad_(True) for t in qkv.split(H * D, dim=-1))
    i = torch.arange(T, device=dev)
    seen = i[None, :] <= i[:, None]
    if band:
        seen &= i[None, :] // 128 > i[:, None] // 128 - band
    p = torch.softmax((q @ k.transpose(-1, -2).contiguous() * D ** -0.5).masked_fill(~seen, float("-inf")), -1)
    (p @ v).backward(do.permute(0, 2, 1, 3).float())
    if tables is None:   # P, dS and each result are rounded once to bf16 (2^-9 relative): their errors add up to less than 1e-2 of a gradient's norm
        for got, want in zip(few.split(H * D, dim=-1), (q, k, v)):
            want = want.grad.permute(0, 2, 1, 3).reshape(1, T, H * D)
            assert ((got.float() - want).norm() / want.norm()).item() < 1e-2


@pytest.mark.parametrize("what", ["inf", "nan"])
def test_pairs_keep_what_is_not_finite_where_it_was(what):
    """A row of dO that is not finite reaches the keys that one wavefront's kernel lets it reach, and no others."""
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(3)
    T, H, D, many = 512, 1, 64, 257
    qkv = torch.randn(1, T, 3 * D, generator=g, device=dev).bfloat16()
    do = torch.randn(1, T, H, D, generator=g, device=dev).bfloat16()
    do[0, 200, 0, 5] = float(what)
    few = _grads(1, T, H, D, 0, None, qkv, do)
    lot = _grads(many, T, H, D, 0, None, qkv.expand(many, -1, -1).contiguous(), do.expand(many, -1, -1, -1).contiguous())
    same = torch.logical_or(few[0] == lot[-1], few[0].isnan() & lot[-1].isnan())
    assert bool(same.all()) and bool(few[0, 256:, D:].isfinite().all())
