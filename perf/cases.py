"""The work that a training program has this package do, as cases that can be timed and compared: whole steps of the
decoder model, evaluation, and the blocks that other training loops call one by one (attention, MLP, experts, loss head,
norms, Newton-Schulz), forward and backward, from the smallest calls to the benchmark's batch.

A case is a dict of plain values; its "kind" says which entry points it runs:

  step            GPT.train_step: forward, backward, AdamW and the fp8 refresh
  eval            GPT.forward without gradients: validation loss
  attention       nki_causal_attention on [B, H, T, D], forward and backward (band: key tiles of a windowed layer, 0 = none)
  rope_attention  nki_rope_attention on the fused [B, T, 3C] projection with its QK norm, forward and backward
  mlp             mlp_fused8 ("fp8"), nr_mlp ("nr": norm and residual folded in) or mlp_fused ("bf16"), forward and backward
  moe             the routed experts, forward and backward (skew: router bias on two experts; experts: "fp8" or "bf16")
  head            norm, LM head and cross entropy, forward and backward
  loss            fused_loss on logits that the caller holds, forward and backward
  rows            the row blocks: rmsnorm_fast, tail_norm2, head_skip, mix_tail, forward and backward
  muon            nsk on a stack of tall and one of wide gradient matrices
"""
import math

import torch

from trainium_frontier_them_bones_amd import autograd as A
from trainium_frontier_them_bones_amd import train_api as api
from trainium_frontier_them_bones_amd.model import GPT, GPTConfig, zipf_tokens

bf16 = torch.bfloat16


def listed():
    return [
        # the benchmark's step: 12 layers, width 768, 16 sequences of 2048 tokens
        _step("step_16x2048", 16, 2048, 12, 768, 64, 32768),
        # the same model on one sequence: a micro-batch of a long accumulation, a run on a small budget, the parity check
        _step("step_1x2048", 1, 2048, 12, 768, 64, 32768),
        # a small model on short ragged sequences with the logit softcap: tests, ablations, sweeps
        _step("step_small_ragged", 3, 384, 4, 512, 128, 8192, softcap=15.0),
        # validation of a width-1024 model with heads of 128 on an odd number of sequences
        dict(_step("eval_5x1920", 5, 1920, 4, 1024, 128, 8192, softcap=15.0), kind="eval"),
        # the benchmark's attention layer
        dict(name="attention_16x12x2048x64", kind="attention", B=16, H=12, T=2048, D=64, band=0),
        # one layer of the width-1024 model with QK norm, heads of 128, a sequence length that is no power of two
        dict(name="rope_attention_3x8x1664x128", kind="rope_attention", B=3, H=8, T=1664, D=128, band=0),
        # the fp8 MLP of the benchmark's configuration 3, all six products in fp8
        dict(name="mlp_fp8_16384", kind="mlp", form="fp8", B=8, T=2048, d=768, F=3072, dw8=True),
        # a folded MLP block on a batch whose rows are no multiple of a tile (padded by the call)
        dict(name="mlp_nr_ragged_1500", kind="mlp", form="nr", B=2, T=750, d=1024, F=4096, dw8=True),
        # the benchmark's loss head alone
        dict(name="head_8192x32768", kind="head", B=4, T=2048, d=768, V=32768, softcap=0.0),
        # the expert layer of configuration 5 with two favoured experts
        dict(name="moe_16384_skewed", kind="moe", B=8, T=2048, d=1024, F=2816, E=8, topk=2, skew=2.0, experts="fp8"),
        # the smallest call: the residual add and norm of one short sequence
        dict(name="rows_tail_norm_256", kind="rows", op="tail_norm2", B=1, T=256, C=768),
        # Muon's orthogonalisation of a model's MLP matrices
        dict(name="muon_12x3072x768", kind="muon", K=12, M=3072, N=768),
    ]


def _step(name, B, T, layers, d, D, V, softcap=0.0):
    return dict(name=name, kind="step", B=B, T=T, layers=layers, d=d, D=D, F=4 * d, V=V, softcap=softcap)


def _log(rng, lo, hi, mult=1):
    """A multiple of mult between lo and hi, spread over the logarithm."""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(max(round(x / mult), -(-lo // mult)), hi // mult)) * mult


def _tokens(rng, most, T_lo, T_hi, T_mult):
    """(B, T): a batch of at most `most` tokens, sequence and batch both spread over their logarithm."""
    T = _log(rng, T_lo, min(T_hi, most), T_mult)
    return _log(rng, 1, max(1, most // T)), T


def draw(rng):
    kind = rng.choice(["step", "eval", "attention", "rope_attention", "mlp", "moe", "head", "loss", "rows", "muon"])
    if kind in ("step", "eval"):
        B, T = _tokens(rng, 16384, 128, 2048, 128)
        D, d = rng.choice([(64, 256), (64, 512), (64, 768), (128, 512), (128, 1024)])
        c = _step("", B, T, rng.choice([2, 3, 4, 6]), d, D, rng.choice([1024, 8192, 32768]), rng.choice([0.0, 15.0]))
        del c["name"]
        return dict(c, kind=kind)
    if kind in ("attention", "rope_attention"):
        B, T = _tokens(rng, 32768, 128, 4096, 128)
        D = rng.choice([64, 128])
        H = rng.choice([2, 4, 6, 8, 12] if D == 64 else [2, 4, 6, 8])
        return dict(kind=kind, B=B, H=H, T=T, D=D, band=rng.choice([0, 0, 0, 2, 4, 8]))
    if kind == "mlp":
        form = rng.choice(["fp8", "nr", "bf16"])
        B, T = _tokens(rng, 32768, 128, 2048, 128) if form == "bf16" else _tokens(rng, 32768, 100, 2048, 1)
        d, F = rng.choice([(512, 2048), (768, 3072), (1024, 4096), (1536, 6144)])
        return dict(kind=kind, form=form, B=B, T=T, d=d, F=F, dw8=rng.choice([True, True, False]))
    if kind == "moe":
        B, T = _tokens(rng, 16384, 128, 2048, 64)
        d, F = rng.choice([(512, 1024), (768, 1536), (1024, 2816)])
        return dict(kind=kind, B=B, T=T, d=d, F=F, E=rng.choice([4, 8]), topk=rng.choice([1, 2, 2]),
                    skew=rng.choice([0.0, 2.0]), experts=rng.choice(["fp8", "fp8", "bf16"]))
    if kind == "head":
        B, T = _tokens(rng, 16384, 128, 2048, 128)
        return dict(kind=kind, B=B, T=T, d=rng.choice([512, 768, 1024]), V=rng.choice([1024, 8192, 32768]),
                    softcap=rng.choice([0.0, 15.0]))
    if kind == "loss":
        B, T = _tokens(rng, 16384, 100, 2048, 1)
        return dict(kind=kind, B=B, T=T, V=rng.choice([1024, 8192, 32768, 50304]), softcap=rng.choice([0.0, 15.0]))
    if kind == "rows":
        B, T = _tokens(rng, 65536, 100, 4096, 1)
        return dict(kind=kind, op=rng.choice(["rmsnorm_fast", "tail_norm2", "head_skip", "mix_tail"]), B=B, T=T,
                    C=rng.choice([256, 512, 768, 1024, 1536]))
    M, N = rng.choice([(512, 512), (768, 768), (2048, 512), (2304, 768), (3072, 768), (2816, 1024), (4096, 1024)])
    return dict(kind="muon", K=rng.randint(1, 12), M=M, N=N)


class _Linear:
    def __init__(self, weight):
        self.weight = weight


class _Mlp:
    """What the MLP calls read of a module: c_fc.weight [F, d] and c_proj.weight [d, F]."""

    def __init__(self, w_fc, w_proj):
        self.c_fc, self.c_proj = _Linear(w_fc), _Linear(w_proj)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)

    def normal(*shape, std=1.0, mean=0.0, dtype=bf16):
        return (torch.randn(*shape, generator=g, device=dev) * std + mean).to(dtype)

    def leaf(*shape, **kw):
        return normal(*shape, **kw).requires_grad_(True)

    s = dict(case)
    kind = case["kind"]
    if kind in ("step", "eval"):
        cfg = GPTConfig(n_layer=case["layers"], d_model=case["d"], n_head=case["d"] // case["D"], d_ff=case["F"],
                        vocab=case["V"], seq_len=case["T"], softcap=case["softcap"])
        s["model"] = GPT(cfg, dev, seed=seed)
        idx, tg = zipf_tokens(case["B"], case["T"], case["V"], seed=seed)
        s["idx"], s["targets"] = idx.to(dev), tg.to(dev)
    elif kind == "attention":
        B, H, T, D = case["B"], case["H"], case["T"], case["D"]
        s["q"], s["k"], s["v"] = leaf(B, H, T, D), leaf(B, H, T, D), leaf(B, H, T, D)
        s["g"] = normal(B, T, H, D)
    elif kind == "rope_attention":
        B, H, T, D = case["B"], case["H"], case["T"], case["D"]
        s["qkv"], s["g"] = leaf(B, T, 3 * H * D), normal(B, T, H, D)
        inv_freq = 10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float32) / D)
        angle = torch.outer(torch.arange(T, dtype=torch.float32), inv_freq)
        s["cos"], s["sin"] = angle.cos().to(bf16).to(dev), angle.sin().to(bf16).to(dev)
    elif kind == "mlp":
        d, F = case["d"], case["F"]
        s["mlp"] = _Mlp(leaf(F, d, std=0.02), leaf(d, F, std=0.02))
        s["x"], s["g"] = leaf(case["B"], case["T"], d), normal(case["B"], case["T"], d)
        if case["form"] != "bf16":
            api.fp8_refresh_weights([s["mlp"]], dw_fp8=case["dw8"])
    elif kind == "moe":
        d, F, E = case["d"], case["F"], case["E"]
        s["h"], s["g"] = leaf(case["B"], case["T"], d), normal(case["B"], case["T"], d)
        s["router"] = leaf(E, d, std=0.02, dtype=torch.float32)
        s["w_fc"], s["w_proj"] = leaf(E, F, d, std=0.02), leaf(E, d, F, std=0.02)
        s["bias"] = torch.tensor([case["skew"]] * 2 + [0.0] * (E - 2), device=dev)
        s["state"] = None
        if case["experts"] == "fp8":
            s["state"] = A.Moe8State(dw_fp8=True)
            s["state"].refresh(s["w_fc"], s["w_proj"])
    elif kind == "head":
        d, V = case["d"], case["V"]
        s["x"], s["w_norm"], s["w_head"] = leaf(case["B"], case["T"], d), leaf(d, std=0.02, mean=1.0), leaf(V, d, std=0.02)
        s["targets"] = torch.randint(0, V, (case["B"], case["T"]), generator=g, device=dev)
    elif kind == "loss":
        V = case["V"]
        s["logits"] = leaf(case["B"], case["T"], V, std=2.0)
        s["targets"] = torch.randint(0, V, (case["B"], case["T"]), generator=g, device=dev)
        s["targets"][:, -1] = -1                                    # the last token of a document has no next one
    elif kind == "rows":
        shape = (case["B"], case["T"], case["C"])
        n_in = {"rmsnorm_fast": 1, "tail_norm2": 2, "head_skip": 3, "mix_tail": 1}[case["op"]]
        s["x"] = [leaf(*shape) for _ in range(n_in)]
        s["gain"] = [leaf(1, std=0.1, mean=m, dtype=torch.float32) for m in (1.0, 0.2, 0.5)]
        s["g"] = [normal(*shape), normal(*shape)]
    elif kind == "muon":
        K, M, N = case["K"], case["M"], case["N"]
        for side, shape in (("a", (K, M, N)), ("b", (K, N, M))):
            grad = normal(*shape, std=0.02, dtype=torch.float32)
            s["g" + side], s["d" + side] = grad, grad.to(bf16).norm(dim=(-2, -1)) * 1.01 + 1e-6
    return s


def run(s):
    kind = s["kind"]
    grad = torch.autograd.grad
    if kind == "step":
        m = s["model"]
        loss = m.train_step(s["idx"], s["targets"])
        return {"loss": loss.detach(), "grad_matrices": m.mats.grad, "grad_others": m.others.grad, "matrices": m.mats.master,
                "others": m.others.master, "matrices_bf16": m.mats.w, "others_bf16": m.others.w, "m_matrices": m.mats.m,
                "m_others": m.others.m, "v_matrices": m.mats.v, "v_others": m.others.v}
    if kind == "eval":
        with torch.no_grad():
            return s["model"].forward(s["idx"], s["targets"])
    if kind == "attention":
        y = api.nki_causal_attention(s["q"], s["k"], s["v"], nw=s["band"])
        return (y.detach(),) + grad(y, (s["q"], s["k"], s["v"]), s["g"])
    if kind == "rope_attention":
        y = api.nki_rope_attention(s["qkv"], s["cos"], s["sin"], s["H"], nw=s["band"])
        return (y.detach(),) + grad(y, (s["qkv"],), s["g"])
    if kind == "mlp":
        call = {"fp8": api.mlp_fused8, "nr": api.nr_mlp, "bf16": api.mlp_fused}[s["form"]]
        y = call(s["mlp"], s["x"])
        return (y.detach(),) + grad(y, (s["x"], s["mlp"].c_fc.weight, s["mlp"].c_proj.weight), s["g"])
    if kind == "moe":
        y = A.MoeMlp8Fn.apply(s["h"], s["router"], s["w_fc"], s["w_proj"], s["state"], s["topk"], s["bias"])
        return (y.detach(),) + grad(y, (s["h"], s["router"], s["w_fc"], s["w_proj"]), s["g"])
    if kind == "head":
        loss = A.LmHeadLossFn.apply(A.RMSNormFn.apply(s["x"], s["w_norm"], 1e-6), s["w_head"], s["targets"], s["softcap"], "mean")
        return (loss.detach(),) + grad(loss, (s["x"], s["w_norm"], s["w_head"]))
    if kind == "loss":
        loss = api.fused_loss(s["logits"], s["targets"], "mean", s["softcap"])
        return (loss.detach(),) + grad(loss, (s["logits"],))
    if kind == "muon":
        return api.nsk(s["ga"], s["gb"], s["da"], s["db"])
    x, (l1, l2, l3), (g1, g2) = s["x"], s["gain"], s["g"]
    if s["op"] == "rmsnorm_fast":
        y = api.rmsnorm_fast(x[0])
        return (y.detach(),) + grad(y, (x[0],), g1)
    if s["op"] == "tail_norm2":
        out, wrt = api.tail_norm2(x[0], x[1]), (x[0], x[1])
    elif s["op"] == "head_skip":
        out, wrt = api.head_skip(x[0], x[1], x[2], l1, l2, l3), (x[0], x[1], x[2], l1, l2, l3)
    else:
        out, wrt = api.mix_tail(x[0], None, l2), (x[0], l2)
    return tuple(t.detach() for t in out) + grad(out, wrt, (g1, g2))


def _seen_keys(T, band):
    """Query-key pairs of one head of a causal sequence; with a band, of the last `band` tiles of 128 keys only."""
    full = T * (T + 1) / 2
    if not band or band * 128 >= T:
        return full
    far = T - band * 128                        # tiles beyond the band, whole ones
    return full - far / 128 * (far / 128 + 1) / 2 * 128 * 128


def work(case):
    kind = case["kind"]
    if kind in ("step", "eval"):
        d, F, V, L, n = case["d"], case["F"], case["V"], case["layers"], case["B"] * case["T"]
        mats, others = L * (4 * d * d + 2 * d * F) + d * V, V * d + (2 * L + 1) * d
        attn = case["B"] * L * (d // case["D"]) * case["D"] * _seen_keys(case["T"], 0)
        if kind == "eval":
            return {"bytes": 2 * (mats + min(n, V) * d) + 16 * n, "flops": 2 * mats * n + 4 * attn}
        # AdamW reads and writes fp32 master, m, v and writes the bf16 copy; gradients leave as bf16 (matrices) and fp32
        return {"bytes": (24 + 2 + 2) * mats + (24 + 2 + 4) * others + 16 * n, "flops": 6 * mats * n + 14 * attn}
    if kind in ("attention", "rope_attention"):
        B, H, T, D = case["B"], case["H"], case["T"], case["D"]
        # q, k, v, y, dy, dq, dk, dv; two products forward, five backward
        return {"bytes": 8 * 2 * B * H * T * D, "flops": 14 * B * H * D * _seen_keys(T, case["band"])}
    if kind in ("mlp", "moe"):
        n, d, F = case["B"] * case["T"], case["d"], case["F"]
        k, E = (case["topk"], case["E"]) if kind == "moe" else (1, 1)
        return {"bytes": 2 * (4 * n * d + 4 * E * d * F), "flops": 12 * k * n * d * F}
    if kind == "head":
        n, d, V = case["B"] * case["T"], case["d"], case["V"]
        return {"bytes": 4 * n * d + 4 * V * d + 8 * n, "flops": 6 * n * d * V}
    if kind == "loss":
        n, V = case["B"] * case["T"], case["V"]
        return {"bytes": 4 * n * V + 8 * n, "flops": 10 * n * V}
    if kind == "rows":
        n = case["B"] * case["T"] * case["C"]
        # inputs and their gradients, outputs and their gradients
        tensors = {"rmsnorm_fast": 4, "tail_norm2": 8, "head_skip": 10, "mix_tail": 6}[case["op"]]
        return {"bytes": 2 * tensors * n, "flops": 20 * n}
    K, M, N = case["K"], case["M"], case["N"]
    return {"bytes": 2 * K * M * N * (4 + 2), "flops": 2 * 5 * K * (4 * M * N * N + 2 * N ** 3)}


def tolerance(case):
    kind = case["kind"]
    if kind == "step":      # fp8 casts through every layer; the second moments square the gradients' differences
        return {"rel": 3e-2, "max": 0.9}
    if kind == "eval":
        return {"rel": 1e-3}
    if kind == "muon":      # five iterations amplify one-ulp differences of the bf16 intermediates
        return {"rel": 2e-2, "max": 0.5}
    if kind in ("mlp", "moe"):
        return {"rel": 5e-3 if case.get("form") == "bf16" or case.get("experts") == "bf16" else 2e-2, "max": 0.5}
    return {"rel": 5e-3, "max": 0.2}
