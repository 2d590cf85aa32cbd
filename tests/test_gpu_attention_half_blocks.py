"""dK and dV with 64 keys a workgroup: the bits of the kernels with 128, over the forms a call may have."""
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


# one block, odd and even numbers of them, heads that are dealt to the XCDs and not, one workgroup for each CU and more (whose first ones run in
# the opposite order), bands of one tile to all
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T,H,band", [(128, 1, 0), (128, 64, 0), (256, 3, 0), (256, 2, 1), (384, 1, 0), (384, 5, 2), (640, 24, 0), (640, 3, 3), (1152, 1, 3),
                                      (1664, 16, 0), (2048, 11, 0), (2048, 16, 0), (2048, 8, 1), (2048, 8, 4), (2048, 1, 16), (4096, 2, 8)])
def test_half_blocks_have_the_bits_of_whole_ones(T, H, band, D):
    dev = torch.device("cuda:0")
    many = -(-4 * 256 * 128 // (T * H))   # 1024 blocks or more
    assert [_lib.lib().tfb_attn_bwd_pairs_applies(3, n, H, T, D, band) == 0 for n in (1, many)] == [True, False]
    g = torch.Generator(device=dev).manual_seed(T + H + band)
    qkv = torch.randn(1, T, 3 * H * D, generator=g, device=dev).bfloat16()
    do = torch.randn(1, T, H, D, generator=g, device=dev).bfloat16()
    tables = None
    if H % 2 and D == 64:
        from oracle import attention as O
        tables = tuple(t.to(dev) for t in O.rope_tables(T, D))
    few = _grads(1, T, H, D, band, tables, qkv, do)
    lot = _grads(many, T, H, D, band, tables, qkv.expand(many, -1, -1).contiguous(), do.expand(many, -1, -1, -1).contiguous())
    assert torch.equal(few[0], lot[0]) and torch.equal(few[0], lot[-1])
