"""Entry points called through the C-ABI, above all those whose outputs have more rows than their inputs: what they write equals the
plain forms on the given rows bit for bit and is zero beyond, whatever the output buffers held."""
import pytest
import torch

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


def _nan(*shape, dev):
    return torch.full(shape, float("nan"), dtype=bf16, device=dev)


def _p(t):
    return None if t is None else t.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("rows,rows_out", [(1, 128), (127, 128), (129, 256), (300, 300)])
@pytest.mark.parametrize("C", [64, 768, 1544])
@pytest.mark.parametrize("res,want_y", [(False, True), (True, True), (False, False)])
def test_norm_with_padded_rows(dev, rows, rows_out, C, res, want_y):
    from trainium_frontier_them_bones_amd import _lib, ops
    g = torch.Generator().manual_seed(rows + C)
    x, r, w = (torch.randn(*s, generator=g).to(bf16).to(dev) for s in ((rows, C), (rows, C), (C,)))
    r = r if res else None
    s, y, inv, y8 = ops.rmsnorm_fwd_q(x, w, 1e-6, r, 4.0)
    so = torch.empty_like(x) if res else None
    yo = _nan(rows_out, C, dev=dev) if want_y else None
    io = torch.empty(rows, device=dev)
    bo = torch.full((rows_out, C), 0xff, dtype=torch.uint8, device=dev)
    _lib.call("tfb_rmsnorm_fwd_q_pad", _p(x), _p(r), _p(w), _p(so), _p(yo), _p(io), _p(bo), 4.0, rows, rows_out, C, 1e-6, _stream())
    assert torch.equal(io, inv) and torch.equal(bo[:rows], y8) and not bool(bo[rows:].any())
    if want_y:
        assert torch.equal(yo[:rows], y) and not bool(yo[rows:].any())
    if res:
        assert torch.equal(so, s)


@pytest.mark.parametrize("n,n_out", [(8, 16), (2040, 4096), (4096, 4096), (300 * 264, 384 * 264)])
@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("copy", [True, False])
def test_cast_with_padded_rows(dev, n, n_out, fmt, copy):
    from trainium_frontier_them_bones_amd import _lib, ops
    x = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(bf16).to(dev)
    want = ops.quant_fp8(x, 4.0, fmt)
    out = torch.full((n_out,), 0xff, dtype=torch.uint8, device=dev)
    cp = _nan(n_out, dev=dev) if copy else None
    _lib.call("tfb_quant_fp8_pad", _p(x), None, 4.0, fmt, _p(out), _p(cp), n, n_out, _stream())
    assert torch.equal(out[:n], want) and not bool(out[n:].any())
    if copy:
        assert torch.equal(cp[:n], x) and not bool(cp[n:].any())


@pytest.mark.parametrize("rows", [1, 127, 129, 255, 256])
def test_mlp_with_a_residual_of_fewer_rows(dev, rows):
    """The residual is read on its own rows only (it ends with them: what follows is another tensor)."""
    from trainium_frontier_them_bones_amd import _lib, ops
    d, F, M = 256, 512, (rows + 127) // 128 * 128
    g = torch.Generator().manual_seed(rows)
    wf, wp = ((0.05 * torch.randn(*s, generator=g)).to(bf16).to(dev) for s in ((F, d), (d, F)))
    row = ops.mlp8_forward_scales(wf, wp)
    w8 = ops.mlp8_precast(wf, wp, row)
    x8 = ops.quant_fp8(torch.nn.functional.pad(torch.randn(rows, d, generator=g), (0, 0, 0, M - rows)).to(bf16).to(dev), 4.0)
    res = torch.randn(rows, d, generator=g).to(bf16).to(dev)
    y, r, h8 = _nan(M, d, dev=dev), _nan(M, F, dev=dev), torch.empty(M, F, dtype=torch.uint8, device=dev)
    _lib.call("tfb_mlp8_fwd_res_rows", _p(x8), _p(w8), _p(row), _p(res), _p(y), _p(r), _p(h8), M, rows, d, F, _stream())
    plain, r0 = ops.mlp8_fwd(None, w8, row, F, x8=x8)
    assert torch.equal(r, r0) and torch.equal(y[:rows], plain[:rows] + res)


@pytest.mark.parametrize("topk", [1, 2])
@pytest.mark.parametrize("N", [1, 65, 1000])
def test_expert_gradient_bytes_without_the_bf16_rows(dev, N, topk):
    """tfb_moe_quant_dout against the cast of the rows that the combine's backward writes, the padding rows between the
    experts' segments among them."""
    from trainium_frontier_them_bones_amd import _lib, ops
    d, Fd, E = 256, 512, 8
    g = torch.Generator().manual_seed(N)
    h = torch.randn(N, d, generator=g).to(bf16).to(dev)
    router = (0.2 * torch.randn(E, d, generator=g)).to(dev)
    rows = torch.stack([ops.mlp8_forward_scales((0.02 * torch.randn(Fd, d, generator=g)).to(bf16).to(dev),
                                                (0.02 * torch.randn(d, Fd, generator=g)).to(bf16).to(dev)) for _ in range(E)])
    _, idx, gate, _ = ops.moe_route(h, router, topk)
    tab = ops.moe_tables(idx, E)
    ys = torch.randn(tab["rmax"], d, generator=g).to(bf16).to(dev)
    dout = torch.randn(N, d, generator=g).to(bf16).to(dev)
    dys, _, rowmax = ops.moe_combine_bwd(dout, ys, tab, gate, want_rowmax=True)
    rows_b = ops.moe_backward_scales_rowmax(rowmax, rows, tab, d)
    out = torch.full((tab["rmax"], d), 0xff, dtype=torch.uint8, device=dev)
    _lib.call("tfb_moe_quant_dout", _p(dout), _p(tab["tok"]), _p(tab["ksel"]), _p(gate), _p(tab["tile_expert"]), _p(rows_b), 5,
              _p(out), tab["rmax"], d, topk, _stream())
    used = int(tab["seg"][-1])
    assert torch.equal(out[:used], ops.moe_quant(dys, rows_b, 5, ops.FMT_E5M2, tab)[:used])


@pytest.mark.parametrize("n,V", [(1, 8), (1000, 512), (5000, 32768), (300, 50304)])
def test_embedding_backward_stays_within_the_scratch_it_asks_for(dev, n, V):
    """tfb_embedding_bwd_grouped with exactly tfb_embedding_bwd_scratch_ints ints, a guard behind them, against the op."""
    from trainium_frontier_them_bones_amd import _lib, ops
    g = torch.Generator().manual_seed(n)
    idx = torch.randint(0, V, (n,), generator=g).to(dev)
    dy = torch.randn(n, 64, generator=g).to(bf16).to(dev)
    ints = int(_lib.lib().tfb_embedding_bwd_scratch_ints(n, V))
    scr = torch.full((ints + 64,), 0x5a5a5a5a, dtype=torch.int32, device=dev)
    dw, want = torch.zeros(V, 64, device=dev), torch.zeros(V, 64, device=dev)
    _lib.call("tfb_embedding_bwd_grouped", _p(idx), 1, _p(dy), _p(dw), n, 64, V, _p(scr), _stream())
    ops.embedding_bwd(idx, dy, want)
    assert torch.equal(scr[ints:], torch.full_like(scr[ints:], 0x5a5a5a5a))
    assert torch.equal(want, dw) or (want - dw).norm() < 1e-6 * want.norm()
