"""tfb_ns5, which takes the reciprocals that its caller computed, against tfb_ns5_stacks, which takes the denominators."""
import ctypes

import pytest
import torch

from trainium_frontier_them_bones_amd import _lib, ops

pytestmark = pytest.mark.gpu


# tall and wide, square; tiles of 64 x 64 and of 128 x 128 in the symmetric products
@pytest.mark.parametrize("K,r,c", [(1, 128, 128), (3, 512, 256), (2, 256, 384), (40, 384, 384), (9, 640, 1152)])
def test_ns5_has_the_bits_of_ns5_stacks(K, r, c):
    dev = torch.device("cuda:0")
    g = torch.randn(K, r, c, generator=torch.Generator(device=dev).manual_seed(K + r + c), device=dev) * 0.02
    d = g.norm(dim=(-2, -1)) * 1.01
    M, N = max(r, c), min(r, c)
    y, v = torch.full((K, r, c), float("nan"), dtype=torch.bfloat16, device=dev), torch.full((K, M), float("nan"), device=dev)
    inv = 1.0 / d
    need = _lib.lib().tfb_ns5_workspace_bytes(K, M, N)
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    co = (ctypes.c_float * 15)(*[x for t in ops.NS_COEFFS for x in t])
    args = [g.data_ptr(), inv.data_ptr(), co, y.data_ptr(), v.data_ptr(), K, M, N, int(r < c), ws.data_ptr()]
    stream = torch.cuda.current_stream().cuda_stream
    assert _lib.lib().tfb_ns5(*args, need - 1, stream) == 4   # (a workspace too small: refused, nothing written)
    _lib.call("tfb_ns5", *args, need, stream)
    (y2, v2), = ops.ns5_stacks([(g, d)])
    assert torch.equal(y, y2) and torch.equal(v, v2)
