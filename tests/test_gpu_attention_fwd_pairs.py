"""The forward by pairs of wavefronts: the bits of one wavefront to 32 queries, over the forms a call may have."""
import pytest
import torch

from trainium_frontier_them_bones_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _applies(n, H, T, D, band):
    return _lib.lib().tfb_attn_fwd_pairs_applies(n, H, T, D, band) == 0


# one, two and more blocks of 64 queries, odd and even numbers of tiles, heads that are dealt to the XCDs and not, one workgroup for each CU and
# more, bands of one tile to all; keys that grow along the sequence, so that the reference point moves at every tile, and that do not
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T,H,band,growth", [(128, 1, 0, 0.0), (256, 3, 0, 4.0), (256, 2, 1, 0.0), (384, 5, 2, 1.0), (640, 24, 0, 1.0), (640, 3, 3, 8.0),
                                             (1152, 1, 3, 0.0), (1664, 16, 0, 2.0), (2048, 11, 0, 0.0), (2048, 8, 4, 4.0), (2048, 1, 16, 8.0), (4096, 2, 0, 1.0)])
@pytest.mark.parametrize("layout", ["bhtd", "bthd"])
def test_pairs_have_the_bits_of_one(T, H, band, growth, layout, D):
    dev = torch.device("cuda:0")
    many = -(-4 * 256 * 128 // (T * H))   # 1024 blocks or more
    longest = min(band or T // 128, T // 128)
    assert [_applies(n, H, T, D, band) for n in (1, many)] == [D == 64 or longest > 1, False]
    g = torch.Generator(device=dev).manual_seed(T + H + band)
    shape = (1, H, T, D) if layout == "bhtd" else (1, T, H, D)
    q, k, v = (torch.randn(*shape, generator=g, device=dev) for _ in range(3))
    ramp = 1.0 + growth * torch.arange(T, device=dev) / T
    k = k * (ramp[:, None] if layout == "bhtd" else ramp[:, None, None])
    q, k, v = (t.bfloat16() for t in (q, k, v))
    kw = {"band": band} if band else {}
    few = ops.attn_fwd(q, k, v, D ** -0.5, layout=layout, **kw)
    lot = ops.attn_fwd(*(t.expand(many, -1, -1, -1).contiguous() for t in (q, k, v)), D ** -0.5, layout=layout, **kw)
    for a, b in zip(few, lot):
        assert torch.equal(a[0], b[0]) and torch.equal(a[0], b[-1])
    q, k, v = (t.double() if layout == "bhtd" else t.double().transpose(1, 2) for t in (q, k, v))
    i = torch.arange(T, device=dev)
    seen = i[None, :] <= i[:, None]
    if band:
        seen &= i[None, :] // 128 > i[:, None] // 128 - band
    s = (q @ k.transpose(-1, -2).contiguous() * D ** -0.5).masked_fill(~seen, float("-inf"))
    want = (torch.softmax(s, -1) @ v).transpose(1, 2)
    # P and the result are rounded once to bf16
    assert ((few[0].double().view(want.shape) - want).norm() / want.norm()).item() < 2 * 2.0 ** -8
    assert (few[1].double().view(s.shape[:3]) - torch.logsumexp(s, -1)).abs().max().item() < 1e-2   # (P's rounding moves the row sum by 2^-9 at most)
