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


# the clamped square of the up-projection, read through a second GEMM that is the identity: a power of two as the clamp's scale (one multiplication
# and the scale in the conversion), one that is not, sums beyond the clamp, infinite and tiny ones
@pytest.mark.parametrize("times", [1.0, 0.75])
@pytest.mark.parametrize("M", [128, 16384])
def test_clamped_square_of_the_up_projection(M, times):
    dev = torch.device("cuda:0")
    d, F = (256, 256) if M == 128 else (1024, 2048)
    g = torch.Generator(device=dev).manual_seed(M)
    w_fc = (torch.randn(F, d, generator=g, device=dev) * d ** -0.5).bfloat16()
    w_proj = torch.zeros(d, F, device=dev, dtype=torch.bfloat16)
    w_proj[:, :d] = torch.eye(d, device=dev).bfloat16()
    row = ops.mlp8_forward_scales(w_fc, w_proj)
    w8 = ops.mlp8_precast(w_fc, w_proj, row)
    row[2] *= times                                                  # c
    x = torch.randn(M, d, generator=g, device=dev) * torch.logspace(-6, 2, M, device=dev)[:, None]
    y, r = ops.mlp8_fwd(x.bfloat16(), w8, row, F)[:2]
    rc = (r.float() * row[2]).bfloat16().float().clamp(max=15.375)
    h8 = (rc * rc).to(torch.float8_e4m3fn).float()
    one = w8[2].view(torch.float8_e4m3fn).float().view(d, F)[0, 0]   # the identity's entries as cast
    assert torch.equal(y, (h8[:, :d] * one * row[4]).bfloat16())
