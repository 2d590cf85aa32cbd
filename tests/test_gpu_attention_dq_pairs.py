"""dQ by pairs of wavefronts: the bits of one wavefront to 32 queries (whole launches are compared with the key and value gradients'), also where
an operand is not finite: a pair's second half may not reach queries in front of it."""
import pytest
import torch

from trainium_frontier_them_bones_amd import ops

pytestmark = pytest.mark.gpu


# a key in the first and in the second half of a tile, of a workgroup's own tile and of one before; the last key of all
@pytest.mark.parametrize("key", [70, 100, 250, 383])
@pytest.mark.parametrize("which", [1, 2])   # K or V
@pytest.mark.parametrize("D", [64, 128])
def test_query_gradients_in_pairs_keep_what_is_not_finite_where_it_was(D, which, key):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(key)
    T, many = 384, 343   # three blocks of 128 queries; some 1029, beyond the pairs
    qkv = torch.randn(1, T, 3, 1, D, generator=g, device=dev).bfloat16()
    qkv[0, key, which, 0, 3] = float("inf")
    do = torch.randn(1, T, 1, D, generator=g, device=dev).bfloat16()
    grads = []
    for n in (1, many):
        q, k, v = qkv.expand(n, -1, -1, -1, -1).contiguous().unbind(2)
        o, lse = ops.attn_fwd(q, k, v, D ** -0.5, layout="bthd")
        out = torch.full((n, T, 3, 1, D), float("nan"), device=dev, dtype=torch.bfloat16)
        dq, dk, dv = out.unbind(2)
        ops.attn_bwd(q, k, v, o, do.expand(n, -1, -1, -1).contiguous(), lse, D ** -0.5, "bthd", dq, dk, dv, "bthd")
        grads.append(out)
    few, lot = grads[0][0], grads[1][-1]
    assert bool(torch.logical_or(few == lot, few.isnan() & lot.isnan()).all())
    # the forward pass multiplies whole tiles of 64 keys (0 x inf where they are masked): queries in front of the key's tile are the ones untouched
    assert bool(few[:key // 64 * 64, 0].isfinite().all())
