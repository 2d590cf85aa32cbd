"""The scale row of an fp8 MLP backward and the gradient's bytes at its scale in one launch: the bits of the two calls."""
import pytest
import torch

from trainium_frontier_them_bones_amd import _lib, ops

pytestmark = pytest.mark.gpu


# one workgroup, a part of one, rows up to the next whole tile as zeros, more work than the launch has workgroups; the maxima given (one,
# more than a workgroup has threads) or made; an all-zero gradient, an infinite and a NaN element
SMALL, LARGE = [(1, 128, 256), (128, 128, 256), (1500, 1536, 1024), (300, 384, 768)], [(16384, 16384, 768), (9000, 9088, 1536)]


@pytest.mark.parametrize("special,rows,M,d", [(None, *s) for s in SMALL + LARGE] + [(v, *s) for v in (0.0, float("inf"), float("nan")) for s in SMALL])
@pytest.mark.parametrize("parts", [0, 1, 700])
def test_scaled_gradient_in_one_launch(rows, M, d, parts, special):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(rows + d)
    dy = (3e-4 * torch.randn(rows, d, generator=g, device=dev)).bfloat16()
    if special is not None:
        dy[:, :] = 0.0 if special == 0.0 else dy
        dy[rows // 2, d // 3] = special
    w = torch.randn(256, 256, generator=g, device=dev).bfloat16()
    row = ops.mlp8_forward_scales(w, w)
    amax = None
    if parts:
        m = dy.float().nan_to_num(0.0, float("inf")).abs().flatten()
        amax = torch.zeros(parts, device=dev)
        amax[parts // 2] = m.max()
    stream = torch.cuda.current_stream().cuda_stream
    want_row = torch.empty(16, device=dev)
    scr = torch.empty(4096, device=dev)
    if parts:
        _lib.call("tfb_mlp8_backward_scales_part", amax.data_ptr(), parts, row.data_ptr(), want_row.data_ptr(), d, stream)
    else:
        _lib.call("tfb_mlp8_backward_scales", dy.data_ptr(), row.data_ptr(), want_row.data_ptr(), scr.data_ptr(), rows, d, stream)
    n, n_out = rows * d, M * d
    want8, want_c = torch.empty(M, d, dtype=torch.uint8, device=dev), torch.empty(M, d, dtype=torch.bfloat16, device=dev)
    _lib.call("tfb_quant_fp8_pad", dy.data_ptr(), want_row[5:].data_ptr(), 0.0, 1, want8.data_ptr(), want_c.data_ptr(), n, n_out, stream)
    for copy in (False, True):
        got_row = torch.full((16,), -1.0, device=dev)
        got8, got_c = torch.full_like(want8, 77), torch.full_like(want_c, -7.0)
        _lib.call("tfb_mlp8_backward_quant", dy.data_ptr(), amax.data_ptr() if parts else None, parts, scr.data_ptr(), row.data_ptr(), got_row.data_ptr(),
                  got8.data_ptr(), got_c.data_ptr() if copy else None, n, n_out, d, stream)
        assert torch.equal(got_row.view(torch.int32), want_row.view(torch.int32)) and torch.equal(got8, want8)
        if copy:
            assert torch.equal(got_c.view(torch.int16), want_c.view(torch.int16))
