"""The persistent kernel's narrow output tiles (192 x 256, 256 x 192): the bits of the kernels that smaller calls take."""
import pytest
import torch

from trainium_frontier_them_bones_amd import ops

pytestmark = pytest.mark.gpu

# rows, width, contraction: 192 x 256 in part of a round with slow rows no multiple of 8, in two full rounds; 256 x 192 in one round, in two
# with a ragged last one; contractions of two, three and more k-tiles (64 bf16, 128 fp8 elements)
SHAPES = [(16128, 768, 2), (16384, 768, 3), (32768, 768, 3), (9600, 1024, 2), (12672, 768, 3), (30336, 768, 2), (24192, 1024, 5)]


def _operands(M, N, K, fp8):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a, b, res = (torch.randn(*s, generator=g, device=dev).bfloat16() for s in ((M, K), (N, K), (M, N)))
    if not fp8:
        return a, b, res
    return a.to(torch.float8_e4m3fn).view(torch.uint8), b.to(torch.float8_e4m3fn).view(torch.uint8), res


def _check(call, a, res, exact):
    """The call on all rows against calls on 1024 rows at a time (launches of few tiles: other kernels), and against 64 bits."""
    got = call(a, res)
    for r in range(0, a.size(0), 1024):
        assert torch.equal(got[r:r + 1024], call(a[r:r + 1024], res[r:r + 1024])), r
    want = exact()
    # one or two roundings to 8 bits of mantissa of sums of products that are exact in fp32
    assert ((got[-640:].double() - want).norm() / want.norm()).item() < 2.0 ** -8


@pytest.mark.parametrize("M,N,kt", SHAPES)
@pytest.mark.parametrize("form", ["nt", "nn", "fp8"])
def test_narrow_tile(M, N, kt, form):
    K = kt * (128 if form == "fp8" else 64)
    a, b, res = _operands(M, N, K, form == "fp8")
    if form == "fp8":
        fa, fb = (t.view(torch.float8_e4m3fn).double() for t in (a[-640:], b))
        _check(lambda x, r: ops.gemm_fp8(x, b, dq=0.25), a, res, lambda: fa @ fb.t() * 0.25)
    elif form == "nt":
        _check(lambda x, r: ops.matmul(x, b, trans_b=True), a, res, lambda: a[-640:].double() @ b.double().t())
    else:
        bt = b.t().contiguous()
        _check(lambda x, r: ops.matmul(x, bt), a, res, lambda: a[-640:].double() @ b.double().t())


@pytest.mark.parametrize("M,N", [(12288, 768), (9600, 1024), (32768, 768)])
@pytest.mark.parametrize("fp8", [True, False])
def test_narrow_tile_with_a_residual(M, N, fp8):
    K = 24 * (128 if fp8 else 64)
    a, b, res = _operands(M, N, K, fp8)
    if fp8:
        fa, fb = (t.view(torch.float8_e4m3fn).double() for t in (a[-640:], b))
        _check(lambda x, r: ops.gemm_fp8_res(x, b, r, dq=0.125), a, res, lambda: fa @ fb.t() * 0.125 + res[-640:].double())
    else:
        _check(lambda x, r: ops.matmul_res(x, b, r, trans_b=True), a, res, lambda: a[-640:].double() @ b.double().t() + res[-640:].double())
