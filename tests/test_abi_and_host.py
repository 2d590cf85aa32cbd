"""CPU-side checks: the C-ABI library loads and exports every symbol the header declares (no compute calls), the Python
binding table matches the header, and the host-side model plumbing (flat parameter groups, token generator, FLOP
count) behaves."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "tfb_kernels.h")


def _declared():
    src = open(HEADER).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    decls = {}
    for m in re.finditer(r"\b(int|long)\s+(tfb_\w+)\s*\(([^;]*?)\)\s*;", src, flags=re.S):
        args = [a.strip() for a in m.group(3).split(",") if a.strip() and a.strip() != "void"]
        decls[m.group(2)] = (m.group(1), args)
    return decls


def test_header_declares_entry_points():
    d = _declared()
    assert len(d) >= 25
    for name in ("tfb_gemm_bf16", "tfb_attn_fwd", "tfb_attn_bwd", "tfb_mlp8_fwd", "tfb_mlp8_bwd", "tfb_lmhead_fwd",
                 "tfb_rmsnorm_fwd", "tfb_loss_bwd", "tfb_adamw"):
        assert name in d


def test_library_exports_every_declared_symbol():
    from trainium_frontier_them_bones_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built (run __graft_entry__.build())")
    L = ctypes.CDLL(_lib.LIB_PATH)
    for name in _declared():
        assert hasattr(L, name), name


def test_binding_table_matches_header():
    from trainium_frontier_them_bones_amd import _lib
    d = _declared()
    assert set(_lib.SIGNATURES) == set(d)
    for name, (ret, args) in d.items():
        sig = _lib.SIGNATURES[name]
        assert len(sig) == len(args), name
        for a, c in zip(args, sig):
            if "*" in a:
                assert c in (ctypes.c_void_p, _lib._lp, _lib._fp), (name, a)
            elif a.startswith("float"):
                assert c is ctypes.c_float, (name, a)
            elif a.startswith("long"):
                assert c is ctypes.c_long, (name, a)
            else:
                assert c is ctypes.c_int, (name, a)


def test_ops_refuse_cpu_tensors():
    from trainium_frontier_them_bones_amd import ops
    with pytest.raises(RuntimeError):
        ops.matmul(torch.zeros(128, 64, dtype=torch.bfloat16), torch.zeros(64, 128, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError):
        ops.rmsnorm_fwd(torch.zeros(4, 64, dtype=torch.bfloat16))


def test_flat_params_layout_and_tokens():
    from trainium_frontier_them_bones_amd.model import FlatParams, GPTConfig, zipf_tokens
    fp = FlatParams({"a": (3, 5), "b": (7,), "c": (2, 8)}, torch.float32, "cpu")
    assert fp.offsets["a"] == (0, 15) and fp.offsets["b"][0] == 16 and fp.offsets["c"][0] == 24 and fp.numel == 40
    fp.load("b", torch.arange(7.0))
    assert torch.equal(fp.params["b"].detach().float(), torch.arange(7.0)) and fp.master[16:23].tolist() == list(range(7))
    assert fp.params["a"].grad_buf.shape == (3, 5) and fp.params["a"].grad_buf.dtype == torch.float32
    x, y = zipf_tokens(4, 64, 1000, seed=1)
    x2, _ = zipf_tokens(4, 64, 1000, seed=1)
    assert torch.equal(x, x2) and torch.equal(x[:, 1:], y[:, :-1]) and int(x.max()) < 1000
    cnt = torch.bincount(zipf_tokens(64, 512, 1000, seed=2)[0].reshape(-1), minlength=1000)
    assert cnt[0] > cnt[10] > cnt[200]            # Zipfian: low ids dominate
    cfg = GPTConfig()
    assert cfg.head_dim == 64


def test_bench_flop_formula():
    import bench
    from trainium_frontier_them_bones_amd.model import GPTConfig
    assert abs(bench.flops_per_token(GPTConfig()) / 1e6 - 773.8) < 0.5    # 773.8 MFLOP/token -> 25.36 TFLOP per 32768-token step


def test_every_entry_point_is_reached_from_the_host_layer():
    """Each exported kernel entry point is called by the package's host code (ops / autograd / the reference-named layers)
    or, for the plain forwarding forms, by a test: nothing in the header is dead."""
    import glob
    import os
    from trainium_frontier_them_bones_amd import _lib
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    host = "".join(open(f).read() for f in glob.glob(os.path.join(root, "trainium_frontier_them_bones_amd", "*.py"))
                   if not f.endswith("_lib.py"))
    tests = "".join(open(f).read() for f in glob.glob(os.path.join(root, "tests", "test_gpu_*.py")))
    for name in _lib.SIGNATURES:
        assert ('"%s"' % name) in host or ("." + name + "(") in host or name in tests, name


def test_amax_hint_is_void_after_an_in_place_update():
    """The amax partials a producer hangs on a gradient tensor are used only while the tensor still holds what they were
    taken from: the same memory, and no in-place write since (autograd may accumulate a second gradient into it)."""
    import torch
    from trainium_frontier_them_bones_amd import autograd as A
    t = torch.randn(8, 4)
    am = torch.tensor([float(t.abs().max())])
    A._attach_amax(t, am)
    assert A._amax_hint(t, t.reshape(8, 4)) is am
    assert A._amax_hint(t, t.clone()) is None                 # a copy is other memory
    old = A.USE_AMAX_HINT
    A.USE_AMAX_HINT = False
    try:
        assert A._amax_hint(t, t) is None
    finally:
        A.USE_AMAX_HINT = old
    t.add_(1.0)
    assert A._amax_hint(t, t) is None                         # written to since: the partials are void
    assert A._amax_hint(torch.randn(3), torch.randn(3)) is None


def test_every_entry_point_rejects_null_pointers_and_empty_shapes_on_the_host():
    """Argument checks come before any device work: with every pointer NULL an entry point answers "bad argument" (or
    "unsupported shape" where the sizes are looked at first), and with dummy non-null pointers and all sizes zero it answers
    with one of the two as well; no call reaches a kernel launch (status 3), so this runs without a GPU."""
    import ctypes
    from trainium_frontier_them_bones_amd import _lib
    L = _lib.lib()
    plain = _lib._LONG_RESULT | {"tfb_norm_bwd_blocks", "tfb_resmix_bwd_blocks"}      # size queries: no status to check
    for name, sig in _lib.SIGNATURES.items():
        if name in plain:
            continue
        for null in (True, False):
            args = []
            for t in sig:
                if t is _lib._vp:
                    args.append(None if null else 0x1000)          # never dereferenced on the host
                elif t is _lib._lp:
                    args.append(None if null else (ctypes.c_long * 4)())
                elif t is _lib._fp:
                    args.append(None if null else (ctypes.c_float * 16)())
                elif t is _lib._f:
                    args.append(0.0)
                else:
                    args.append(0)
            assert getattr(L, name)(*args) in (1, 2), (name, null)


def test_every_change_of_the_table_of_timed_entry_points_is_told_to_the_native_layer(monkeypatch):
    """The native layer asks for events only while the table holds something: each way to change a dict tells it, before the
    extension is loaded (the state is handed over at the load) and after."""
    from trainium_frontier_them_bones_amd import _lib
    told = []
    monkeypatch.setitem(_lib.native.__dict__, "set_timed", told.append)
    t = _lib.TIMED
    assert not t
    steps = [(lambda: t.__setitem__("a", []), True), (lambda: t.__delitem__("a"), False), (lambda: t.update(a=[], b=[]), True),
             (lambda: t.pop("a"), True), (lambda: t.popitem(), False), (lambda: t.setdefault("c", []), True), (lambda: t.clear(), False),
             (lambda: t.__ior__({"d": []}), True), (lambda: t.pop("nothing", None), True), (lambda: t.clear(), False)]
    for step, want in steps:
        step()
        assert told.pop() is want and not told and bool(t) is want
    monkeypatch.delitem(_lib.native.__dict__, "set_timed")
    t["a"] = []                                            # nothing is loaded for it
    assert "set_timed" not in _lib.native.__dict__
    t.clear()


@pytest.mark.parametrize("E,d,F,rows,one", [
    (8, 512, 1024, 64, False), (8, 512, 1024, 512, True),          # 128 tiles: half a round
    (4, 256, 512, 128, False), (4, 256, 512, 256, False), (4, 256, 512, 1024, True), (2, 256, 256, 256, False), (2, 256, 256, 1024, True),
    (8, 1024, 2816, 64, False), (8, 1024, 2816, 256, True), (8, 1024, 2816, 4096, True),
    (8, 768, 1536, 128, False), (8, 768, 1536, 512, True),         # 288 tiles: a little more than a round
    (16, 512, 1024, 1, True),                                      # exactly one
    (8, 512, 1024, 0, True),                                       # rows not known
    (8, 384, 1024, 4096, False), (8, 512, 1152, 4096, False), (65, 512, 1024, 4096, False)])   # not the kernel's
def test_expert_gradients_run_as_one_launch_where_rows_and_tiles_fill_it(E, d, F, rows, one):
    """The rule on sizes alone (256 CUs where there is no device to ask)."""
    from trainium_frontier_them_bones_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built (run __graft_entry__.build())")
    L = _lib.lib()
    rmax = L.tfb_moe_max_rows(rows * E, E, 1) if rows else 0
    assert (L.tfb_moe_dw8_one_launch_applies(E, d, F, rmax) == 0) == one


# dQ's and dK/dV's kernels by pairs of wavefronts (1, 2) where a launch's longest block sets the time: as many blocks as that holds for (B H T / 128),
# and some more. A band leaves the blocks alike, so few of them fill the chip.
@pytest.mark.parametrize("D,T,nw,counts", [
    (64, 128, 0, [(128, 1), (192, 0)]), (64, 256, 0, [(128, 3), (192, 2), (384, 0)]), (64, 384, 0, [(384, 0)]), (64, 512, 0, [(192, 3), (384, 0)]),
    (64, 1024, 0, [(288, 3), (384, 2), (448, 0)]), (64, 2048, 0, [(384, 3), (512, 2), (576, 0)]), (64, 4096, 0, [(384, 3), (512, 2), (576, 0)]),
    (64, 2048, 1, [(128, 1), (192, 0), (384, 0)]), (64, 2048, 2, [(128, 3), (192, 2), (384, 0)]), (64, 2048, 8, [(192, 3), (256, 2), (320, 0)]),
    (64, 640, 2, [(320, 0)]), (64, 1024, 2, [(192, 2)]), (64, 2048, 16, [(512, 2)]), (64, 2048, 99, [(512, 2)]),
    (128, 128, 0, [(128, 3), (192, 2), (256, 2)]), (128, 256, 0, [(128, 3), (192, 2)]), (128, 1024, 0, [(256, 3), (320, 2)]),
    (128, 2048, 0, [(288, 3), (384, 2)]), (128, 1024, 2, [(128, 3), (192, 2)]), (128, 2048, 8, [(128, 3), (256, 2)]),
    (96, 2048, 0, [(16, 0)]), (64, 2050, 0, [(16, 0)])])
def test_attention_runs_by_pairs_where_the_longest_block_sets_the_time(D, T, nw, counts):
    """The rule on sizes alone (256 CUs where there is no device to ask)."""
    from trainium_frontier_them_bones_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built (run __graft_entry__.build())")
    for blocks, want in counts:
        got = sum(w for w in (1, 2) if _lib.lib().tfb_attn_bwd_pairs_applies(w, 1, blocks * 128 // T, T, D, nw) == 0)
        assert got == want, blocks
