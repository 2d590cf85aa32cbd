"""The grouped embedding backward's segments (8, 16, 32, 64 positions by the number of rows): frequent tokens that run over many of them, rows
that end inside one, ids outside the vocabulary; added to what is there."""
import pytest
import torch

from trainium_frontier_them_bones_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 9, 512, 513, 2048, 2051, 24575, 24576, 24641])
@pytest.mark.parametrize("C,V", [(264, 500), (1032, 50000)])
def test_segments(n, C, V):
    g = torch.Generator().manual_seed(n)
    idx = (torch.rand(n, generator=g) ** 6 * V).long()           # a few tokens have most of the rows
    idx[::7] = idx[0]
    idx[3::11] = V
    idx[5::13] = -2
    dy, dw = torch.randn(n, C, generator=g).bfloat16(), torch.randn(V, C, generator=g)
    ok = (idx >= 0) & (idx < V)
    want = dw.double().index_add_(0, idx[ok], dy[ok].double())
    got = dw.cuda()
    ops.embedding_bwd(idx.cuda(), dy.cuda(), got)
    # sums of m values in 32 bits in some order: errors of at most m 2^-24 of the sum of their magnitudes
    most = int(torch.bincount(idx[ok]).max()) if bool(ok.any()) else 1
    bound = dw.double().abs().index_add_(0, idx[ok], dy[ok].double().abs()) * (most + 1) * 2.0 ** -24
    assert bool(((got.cpu().double() - want).abs() <= bound).all())


@pytest.mark.parametrize("n", [32767, 32768])   # (rows of 512 columns: segments of 32, then of 64)
def test_segments_of_narrower_rows(n):
    test_segments(n, 512, 500)
