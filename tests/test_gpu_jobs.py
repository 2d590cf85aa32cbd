"""Gradients that run as jobs of one launch: the bits of the launches they replace."""
import pytest
import torch

from trainium_frontier_them_bones_amd import _lib, ops

pytestmark = pytest.mark.gpu
WS = 256 << 20


def _ptr(t):
    return t.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream


# a single tile, a ragged number of tiles per XCD, several k ranges, 64-row tiles for one job, for both, for neither, the most tiles;
# refused: k ranges in workgroups of their own (either GEMM), more tiles than the ring takes
REFUSED = [(128, 3072, 768), (4096, 512, 512), (6144, 768, 768), (8192, 2304, 768), (2048, 3072, 1024)]


@pytest.mark.parametrize("M,N,K", [(128, 128, 128), (384, 640, 256), (1152, 1536, 512), (2048, 2304, 768), (2048, 768, 768), (4096, 768, 768),
                                   (3072, 2304, 768)] + REFUSED)
@pytest.mark.parametrize("f32,accumulate", [(0, 0), (1, 1), (0, 1)])
def test_linear_gradients_in_one_launch(M, N, K, f32, accumulate):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    dy, x, w = (torch.randn(*s, generator=g, device=dev).bfloat16() for s in ((M, N), (M, K), (N, K)))
    old = torch.randn(N, K, generator=g, device=dev).to(torch.float32 if f32 else torch.bfloat16)
    L = _lib.lib()
    assert L.tfb_linear_bwd_applies(M, N, K, WS) == ((M, N, K) in REFUSED)
    if (M, N, K) in REFUSED:
        dx = torch.empty_like(x)
        assert L.tfb_linear_bwd(_ptr(dy), _ptr(x), _ptr(w), _ptr(dx), _ptr(old), M, N, K, f32, accumulate, WS, _stream()) == 1
        return
    dw = old.clone()
    dx = torch.empty_like(x)
    assert L.tfb_linear_bwd(_ptr(dy), _ptr(x), _ptr(w), _ptr(dx), _ptr(dw), M, N, K, f32, accumulate, WS, _stream()) == 0
    assert torch.equal(dx, ops.matmul(dy, w))
    want = ops.matmul(dy, x, trans_a=True, out=old.clone() if accumulate else None, accumulate=bool(accumulate), out_dtype=old.dtype)
    assert torch.equal(dw, want)
    exact = dy.double() @ w.double()                     # and against 64 bits: one rounding of sums of up to N products
    assert ((dx.double() - exact).norm() / exact.norm()).item() < 2.0 ** -8


@pytest.mark.parametrize("M,d,F", [(128, 256, 512), (384, 256, 768), (1152, 512, 2048), (1536, 1024, 4096), (2048, 768, 3072), (4096, 512, 2048),
                                   (8192, 768, 3072)])
@pytest.mark.parametrize("f32,accumulate", [(0, 0), (1, 1)])
def test_mlp_gradients_in_one_launch(M, d, F, f32, accumulate):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + d + F)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()  # noqa: E731
    x, dy, w_fc, w_proj = rnd(M, d), rnd(M, d), rnd(F, d, std=0.02), rnd(d, F, std=0.02)
    row = ops.mlp8_forward_scales(w_fc, w_proj)
    w8 = ops.mlp8_precast(w_fc, w_proj, row)
    _, r, x8 = ops.mlp8_fwd(x, w8, row, F, 4.0, True)
    rowb = ops.mlp8_backward_scales(dy, row)
    L = _lib.lib()
    dt = torch.float32 if f32 else torch.bfloat16
    old = [torch.randn(*s, generator=g, device=dev).to(dt) for s in ((F, d), (d, F))]
    dx, _, dp8, hq8, dy8 = ops.mlp8_bwd_q(dy, r, w8, rowb, 240.0, False)
    assert dp8.numel() == hq8.numel() == r.numel() == M * F and dy8.numel() == x8.numel() == dx.numel() == M * d
    want = ops.mlp8_dw8(x8, dp8, hq8, dy8, rowb, 4.0, *([t.clone() for t in old] if accumulate else [None, None]), accumulate=bool(accumulate),
                        out_dtype=dt)
    got = [t.clone() for t in old]
    dx2, dp2, hq2 = torch.empty_like(dx), torch.empty_like(dp8), torch.empty_like(hq8)
    st = L.tfb_mlp8_bwd_dw8(_ptr(dy8), _ptr(r), _ptr(w8), _ptr(rowb), _ptr(dx2), _ptr(dp2), _ptr(hq2), 240.0, _ptr(x8), 4.0, None, _ptr(got[0]),
                            _ptr(got[1]), M, d, F, f32, accumulate, WS, _stream())
    assert st == L.tfb_mlp8_bwd_dw8_applies(M, d, F, WS) == (M > 4096)
    if st:
        return
    assert torch.equal(dx2, dx) and torch.equal(dp2, dp8) and torch.equal(hq2, hq8)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    # the two weight gradients of tfb_mlp8_dw8 are one launch too: each alone
    fc = ops.gemm_fp8_tn(dp8, x8, 1, 0, rowb[7:8], None, 0.25, out_dtype=dt)
    proj = ops.gemm_fp8_tn(dy8, hq8, 1, 0, rowb[5:6], rowb[13:14], 1.0, out_dtype=dt)
    if not accumulate:
        assert torch.equal(want[0], fc) and torch.equal(want[1], proj)


# workspace_bytes fixes the k ranges that the separate calls would be given, so the order of the sums: none, too little for a second range, enough for
# some of those that the contraction would like, and more than enough
@pytest.mark.parametrize("ws_bytes", [0, 1 << 18, 5 << 20, WS])
@pytest.mark.parametrize("M,N,K", [(128, 128, 128), (384, 2304, 768), (2048, 2304, 768), (4096, 768, 768), (6144, 1536, 512), (256, 4096, 256)])
def test_linear_gradients_have_the_bits_of_calls_with_that_workspace(M, N, K, ws_bytes):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    dy, x, w = (torch.randn(*s, generator=g, device=dev).bfloat16() for s in ((M, N), (M, K), (N, K)))
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=dev)
    L = _lib.lib()
    dx, dw = torch.full_like(x, float("nan")), torch.full((N, K), float("nan"), device=dev)
    st = L.tfb_linear_bwd(_ptr(dy), _ptr(x), _ptr(w), _ptr(dx), _ptr(dw), M, N, K, 1, 0, ws_bytes, _stream())
    assert st == L.tfb_linear_bwd_applies(M, N, K, ws_bytes)
    if st:   # (a range count that the ring would have to cut into workgroups of their own)
        return
    for out, a, b, m, n, k, ta in ((dx, dy, w, M, K, N, 0), (dw, dy, x, N, K, M, 1)):
        want = torch.empty_like(out)
        f32 = int(out.dtype == torch.float32)
        assert L.tfb_gemm_bf16(_ptr(a), _ptr(b), _ptr(want), m, n, k, ta, 0, f32, 0, _ptr(ws) if ws_bytes else None, ws_bytes, _stream()) == 0
        assert torch.equal(out, want)


@pytest.mark.parametrize("ws_bytes", [0, 1 << 18, 9 << 20, WS])
@pytest.mark.parametrize("M,d,F", [(128, 256, 512), (2048, 768, 3072), (4096, 512, 2048), (4096, 256, 1024), (12288, 256, 1024)])
def test_mlp_gradients_have_the_bits_of_calls_with_that_workspace(M, d, F, ws_bytes):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + d + F)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()  # noqa: E731
    x, dy, w_fc, w_proj = rnd(M, d), rnd(M, d), rnd(F, d, std=0.02), rnd(d, F, std=0.02)
    row = ops.mlp8_forward_scales(w_fc, w_proj)
    w8 = ops.mlp8_precast(w_fc, w_proj, row)
    _, r, x8 = ops.mlp8_fwd(x, w8, row, F, 4.0, True)
    rowb = ops.mlp8_backward_scales(dy, row)
    L = _lib.lib()
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=dev)
    dx, _, dp8, hq8, dy8 = ops.mlp8_bwd_q(dy, r, w8, rowb, 240.0, False)
    assert dp8.numel() == hq8.numel() == r.numel() == M * F and dy8.numel() == x8.numel() == dx.numel() == M * d
    got = [torch.full(s, float("nan"), device=dev) for s in ((F, d), (d, F))]
    both, one = [torch.empty_like(t) for t in got], [torch.empty_like(t) for t in got]
    dx2, dp2, hq2 = torch.empty_like(dx), torch.empty_like(dp8), torch.empty_like(hq8)
    st = L.tfb_mlp8_bwd_dw8(_ptr(dy8), _ptr(r), _ptr(w8), _ptr(rowb), _ptr(dx2), _ptr(dp2), _ptr(hq2), 240.0, _ptr(x8), 4.0, None, _ptr(got[0]),
                            _ptr(got[1]), M, d, F, 1, 0, ws_bytes, _stream())
    assert st == L.tfb_mlp8_bwd_dw8_applies(M, d, F, ws_bytes) == 0
    assert L.tfb_mlp8_dw8(_ptr(x8), _ptr(dp8), _ptr(hq8), _ptr(dy8), _ptr(rowb), 4.0, _ptr(both[0]), _ptr(both[1]), M, d, F, 1, 0, _ptr(ws), ws_bytes,
                          None, _stream()) == 0
    for out, g8, a8, s_g, s_a, imm, O, D in ((one[0], dp8, x8, rowb[7:8], None, 0.25, F, d), (one[1], dy8, hq8, rowb[5:6], rowb[13:14], 1.0, d, F)):
        assert L.tfb_gemm_fp8_tn(_ptr(g8), 1, _ptr(a8), 0, _ptr(s_g), None if s_a is None else _ptr(s_a), imm, _ptr(out), M, O, D, 1, 0, _ptr(ws),
                                 ws_bytes, _stream()) == 0
    assert torch.equal(dx2, dx) and torch.equal(dp2, dp8) and torch.equal(hq2, hq8)
    for a, b, c in zip(got, both, one):
        assert torch.equal(a, c) and torch.equal(b, c)
