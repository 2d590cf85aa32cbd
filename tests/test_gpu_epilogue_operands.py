"""The persistent kernel's epilogues with an operand of their own (rotation tables, a residual): the bits of the kernels that smaller calls take."""
import pytest
import torch

from trainium_frontier_them_bones_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=g.device).bfloat16()


# rows, tokens of a sequence, width of the rotated and of all columns, contraction: two, three and many k-tiles; part of a round, two rounds of
# which the last is ragged, the last 128 rows by themselves; nothing rotated, all of it; sequences that end inside a tile; and launches of the
# kernels for fewer tiles
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("M,T,rot,N,K", [(128, 128, 256, 384, 64), (1152, 384, 1024, 1536, 512), (6144, 96, 2048, 3072, 128), (16384, 2048, 512, 768, 128), (16384, 512, 768, 768, 192), (20480, 640, 1536, 2304, 128), (28672, 7168, 1024, 1536, 512),
                                         (30336, 1264, 1024, 1536, 128), (12288, 384, 0, 2304, 768), (32768, 2048, 1536, 2304, 768)])
def test_rotated_projection(M, T, rot, N, K, D):
    g = torch.Generator(device="cuda:0").manual_seed(M + N + K)
    x, w, cos, sin = _normal(g, M, K), _normal(g, N, K), _normal(g, T, D // 2), _normal(g, T, D // 2)
    if D == 64:
        got = ops.qkv_rope(x, w, cos, sin, T, rot)
    else:
        got = torch.full((M, N), float("nan"), device=x.device, dtype=torch.bfloat16)
        args = [t.data_ptr() for t in (x, w, cos, sin, got)] + [M, N, K, T, rot, D, torch.cuda.current_stream().cuda_stream]
        assert _lib.lib().tfb_qkv_rope_heads_fwd(*args) == 0
    want = ops.matmul(x, w, trans_b=True)
    if rot:
        ops.rope_(want, cos, sin, T, rot // D, D)
    assert torch.equal(got, want)


# tiles of 256 x 256 in one round and in two, of 192 x 256 and 256 x 192; the last 128 rows by themselves
@pytest.mark.parametrize("M,N", [(16384, 1024), (28672, 1024), (16512, 1024), (12288, 768), (9600, 1024)])
@pytest.mark.parametrize("fp8", [True, False])
def test_residual(M, N, fp8):
    K, g = 24 * (128 if fp8 else 64), torch.Generator(device="cuda:0").manual_seed(M + N)
    a, b, res = _normal(g, M, K), _normal(g, N, K), _normal(g, M, N)
    if fp8:
        a, b = (t.to(torch.float8_e4m3fn).view(torch.uint8) for t in (a, b))
        got, plain = ops.gemm_fp8_res(a, b, res, dq=0.125), ops.gemm_fp8(a, b, dq=0.125)
    else:
        got, plain = ops.matmul_res(a, b, res, trans_b=True), ops.matmul(a, b, trans_b=True)
    assert torch.equal(got, res + plain)
