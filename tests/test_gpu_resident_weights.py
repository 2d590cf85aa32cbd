"""The up-projection and dH kernels that keep the weights in registers: the bits of the tiled kernels, which launches of fewer rows run."""
import pytest
import torch

from trainium_frontier_them_bones_amd import ops

pytestmark = pytest.mark.gpu


# the fewest rows (eight tiles of 64 for each CU and panel of 256), tiles that divide among the XCDs and that do not (K = 1024: tiles of 32
# rows, 128 rows being four; K = 768: 64), a panel border inside a workgroup's run and at its end
@pytest.mark.parametrize("M,d,F", [(8192, 1024, 4096), (8320, 1024, 4096), (11904, 1024, 2816), (32768, 1024, 1024), (11008, 768, 3072), (16384, 768, 2048)])
def test_many_rows_equal_few(M, d, F):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + F)
    w_fc = (torch.randn(F, d, generator=g, device=dev) * d ** -0.5).bfloat16()
    w_proj = (torch.randn(d, F, generator=g, device=dev) * F ** -0.5).bfloat16()
    row = ops.mlp8_forward_scales(w_fc, w_proj)
    w8 = ops.mlp8_precast(w_fc, w_proj, row)
    x = torch.randn(M, d, generator=g, device=dev).bfloat16()
    dy = (1e-3 * torch.randn(M, d, generator=g, device=dev)).bfloat16()
    back = ops.mlp8_backward_scales(dy, row)

    def run(x, dy):
        y, r = ops.mlp8_fwd(x, w8, row, F)[:2]
        dx, _, dp8, hq8, _ = ops.mlp8_bwd_q(dy, r, w8, back, want_dpre=False)
        return y, r, dx, dp8, hq8
    all_rows = run(x, dy)
    for i in (0, M - 1024):
        few = run(x[i:i + 1024].contiguous(), dy[i:i + 1024].contiguous())
        assert all(torch.equal(a[i:i + 1024], b) for a, b in zip(all_rows, few))
    # and every row against its own group of 1024: the tiles of every XCD
    r = torch.cat([ops.mlp8_fwd(c.contiguous(), w8, row, F)[1] for c in x.split(1024)])
    assert torch.equal(all_rows[1], r)
