"""What this framework's users have it do, as cases that can be timed and checked.

A case is a dict of plain values; `kind` names the path and the rest are its sizes:

  eval       a recursive_macro model's logits for a batch of sequences, no gradients
  pool       the routed cluster-pool SwiGLU layer (fp32 master weights), forward + backward
  pool_eval  the same layer without gradients
  block      a dense transformer block (norm, QKV + RoPE + causal attention, norm, SwiGLU), forward + backward
  swiglu     the dense SwiGLU layer; `grad` False is the forward alone
  svd        the SVD low-rank SwiGLU FFN, forward + backward
  head       the LM head with its cross-entropy, forward + backward
  shortlist  the shortlist output head (candidate build, logits, loss), forward + backward
  step       one captured training step of the recursive_macro engine (audit replay, consistency
             and distillation terms, backward, AdamW)

Each kind goes through the entry point a program calls: the layer modules, `hip_ops`, the model
or the engine.  `exact` restates the layers in 64-bit torch; the bf16 paths' operands are bf16 by
contract, so it starts from the operands' bf16 values.
"""

from __future__ import annotations

import sys
from pathlib import Path

import torch
import torch.nn.functional as F
from torch import nn

_PKG = Path(__file__).resolve().parent.parent / "speedup-thingy_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

from rte_amd.config import ExperimentConfig, ModelConfig, OutputConfig, TrainingConfig  # noqa: E402
from rte_amd.kernels import hip_ops  # noqa: E402
from rte_amd.layers import ClusterPoolSwiGLU, DenseSwiGLU, TransformerBlock  # noqa: E402
from rte_amd.models import RecursiveModel  # noqa: E402
from rte_amd.output import ShortlistHead  # noqa: E402
from rte_amd.training import TrainEngine  # noqa: E402

DEV = "cuda"
BF16 = torch.bfloat16
F64 = torch.float64
WIDE = (8192, 2048, 8192)  # tokens, width, neurons of the largest case: drawn ones cost no more

# (d, clusters, neurons per cluster, top-k) of the routed pools in the configurations: the CPU
# baseline layer, the recursive_macro step and the scaled shortlist step
POOLS = ((256, 32, 32, 4), (512, 64, 32, 8), (1024, 256, 64, 16))


# ----------------------------------------------------------------------------- the cases

def listed():
    return [
        # one short sequence through the whole model (what scoring a single prompt costs): launches
        dict(name="eval_1x64", kind="eval", B=1, S=64, d=512),
        # a ragged handful of tokens through one routed layer
        dict(name="pool_eval_333", kind="pool_eval", T=333, d=512, C=64, n=32, k=8),
        # the routed layer of the recursive_macro training step, batch 128 x 64
        dict(name="pool_8192", kind="pool", T=8192, d=512, C=64, n=32, k=8, fp32=False),
        # the routed layer of the scaled step, batch 32 x 512: the largest pool
        dict(name="pool_16384", kind="pool", T=16384, d=1024, C=256, n=64, k=16, fp32=False),
        # the layer in the reference's default precision, at the CPU baseline's sizes
        dict(name="pool_fp32_8192", kind="pool", T=8192, d=256, C=32, n=32, k=4, fp32=True),
        # the dense block of the fused QKV + SwiGLU configuration, batch 128 x 64
        dict(name="block_128x64", kind="block", B=128, S=64, d=512, heads=8, ff=2048),
        # a block at the scaled step's width and sequence length
        dict(name="block_32x512", kind="block", B=32, S=512, d=1024, heads=16, ff=4096),
        # the widest dense FFN layer the reference's kernel reports time
        dict(name="swiglu_2048x8192", kind="swiglu", T=WIDE[0], d=WIDE[1], ff=WIDE[2], grad=True),
        # the SVD low-rank FFN configuration
        dict(name="svd_32768", kind="svd", T=32768, d=1024, ff=4096, r=128),
        # the tied head of the recursive_macro step with its loss
        dict(name="head_8192", kind="head", T=8192, d=512, V=2048),
        # the scaled step's shortlist head
        dict(name="shortlist_32x512", kind="shortlist", B=32, S=512, d=1024, V=8192),
        # the whole recursive_macro training step, batch 128 x 64
        dict(name="step_128x64", kind="step", B=128, S=64, d=512),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(lo * (hi / lo) ** rng.random() + 0.5)))


def draw(rng):
    kind = rng.choice(["eval", "pool", "pool", "pool_eval", "block", "block", "swiglu", "swiglu", "svd", "head",
                       "shortlist", "step"])
    if kind == "eval":
        return dict(kind=kind, B=_spread(rng, 1, 16), S=_spread(rng, 16, 64), d=rng.choice([256, 512]))
    if kind in ("pool", "pool_eval"):
        d, C, n, k = rng.choice(POOLS)
        if kind == "pool_eval":
            return dict(kind=kind, T=_spread(rng, 1, 2048), d=d, C=C, n=n, k=k)
        fp32 = d < 1024 and rng.random() < 0.3
        return dict(kind=kind, T=_spread(rng, 256, 8192 if d < 1024 else 16384), d=d, C=C, n=n, k=k, fp32=fp32)
    if kind == "block":
        d = rng.choice([256, 512, 1024])
        S = _spread(rng, 16, 1024)
        B = max(1, _spread(rng, 1024, 16384) // S)
        return dict(kind=kind, B=B, S=S, d=d, heads=d // rng.choice([32, 64, 64, 128]),
                    ff=32 * _spread(rng, d // 16, d // 8))
    if kind == "swiglu":
        d = rng.choice([512, 1024, 2048])
        return dict(kind=kind, T=_spread(rng, 64, 8192), d=d, ff=32 * _spread(rng, d // 32, d // 8),
                    grad=rng.random() < 0.7)
    if kind == "svd":
        return dict(kind=kind, T=_spread(rng, 1024, 32768), d=rng.choice([512, 1024]), ff=rng.choice([2048, 4096]),
                    r=rng.choice([32, 64, 128]))
    if kind == "head":
        return dict(kind=kind, T=_spread(rng, 128, 8192), d=rng.choice([256, 512, 1024]), V=8 * _spread(rng, 128, 1024))
    if kind == "shortlist":
        S = _spread(rng, 64, 512)
        return dict(kind=kind, B=max(1, _spread(rng, 256, 16384) // S), S=S, d=rng.choice([512, 1024]),
                    V=_spread(rng, 2048, 8192))
    return dict(kind=kind, B=_spread(rng, 16, 128), S=_spread(rng, 24, 64), d=rng.choice([256, 512]))


# ----------------------------------------------------------------------------- programs

def _model_config(d):
    """The recursive_macro model of the training configuration (64 x 32 pools, top-8) at width d."""
    return ModelConfig(
        topology="recursive", vocab_size=2048, d_model=d, n_heads=d // 64, d_ff=2048, n_dense_layers=2, n_prelude=1,
        n_coda=1, t_max=4, depth_choices=[1, 2, 4], attn_banks=1, ffn_banks=1, head_groups=d // 64, ffn_groups=64,
        active_head_groups=2, active_ffn_groups=8, recipe_count=16, macro_rank=32, ffn_kind="cluster_pool",
        ffn_clusters=64, ffn_top_k=8)


def _dense_config(d, ff, heads=None, **pool):
    """The configuration a single layer or block is built from."""
    heads = heads or d // 64
    return ModelConfig(topology="dense", vocab_size=64, d_model=d, n_heads=heads, d_ff=ff, n_dense_layers=1, n_prelude=1,
                       n_coda=1, t_max=1, depth_choices=[1], attn_banks=1, ffn_banks=1, head_groups=1, ffn_groups=1,
                       active_head_groups=1, active_ffn_groups=1, recipe_count=2, **pool)


def _zipf(shape, vocab, g):
    """Token ids with Zipf(1.1) frequencies."""
    p = (torch.arange(vocab, dtype=torch.float32, device=DEV) + 1.0).pow(-1.1)
    n = 1
    for s in shape:
        n *= s
    return torch.multinomial(p, n, replacement=True, generator=g).view(shape)


def _running(module, g):
    """Weights of a run in progress: nothing is left at a zero or one it was initialised to."""
    with torch.no_grad():
        for p in module.parameters():
            p.add_(torch.randn(p.shape, device=p.device, generator=g) * 0.02)


def prepare(case, seed):
    kind = case["kind"]
    torch.manual_seed(seed)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)

    def rnd(*shape):
        return torch.randn(*shape, device=DEV, generator=g)

    s = {"case": case}
    if kind in ("eval", "step"):
        cfg = _model_config(case["d"])
        tokens = _zipf((case["B"], case["S"] + 1), cfg.vocab_size, g)
        s["tokens"], s["targets"] = tokens[:, :-1].contiguous(), tokens[:, 1:].contiguous()
        if kind == "eval":
            with torch.device(DEV):
                s["model"] = RecursiveModel(cfg, OutputConfig())
            _running(s["model"], g)
            s["recipe"] = seed % cfg.recipe_count
            return s
        tr = TrainingConfig(mode="recursive_macro", precision="bf16", lr=3e-4, weight_decay=0.1, batch_size=case["B"],
                            seq_len=case["S"], audit_sampler="fixed_count", audit_fixed_count=1, fixed_depth=4,
                            seed=seed)
        with torch.device(DEV):
            model = RecursiveModel(cfg, OutputConfig())
        _running(model, g)
        eng = TrainEngine(ExperimentConfig(model=cfg, training=tr, output=OutputConfig(), run_name="step"),
                          device=torch.device(DEV), recursive_model=model)
        eng.enable_graph_capture()
        for _ in range(3):  # two eager steps and the captured one: a program makes them once
            eng.train_step((s["tokens"], s["targets"]))
        s["engine"] = eng
        return s
    if kind in ("pool", "pool_eval"):
        d = case["d"]
        with torch.device(DEV):
            s["layer"] = ClusterPoolSwiGLU(_dense_config(d, case["C"] * case["n"], ffn_kind="cluster_pool",
                                                         ffn_clusters=case["C"], ffn_top_k=case["k"]))
        x = rnd(case["T"], d)
        fp32 = bool(case.get("fp32"))
        s["x"] = (x if fp32 else x.to(BF16)).requires_grad_(kind == "pool")
        s["dy"] = rnd(case["T"], d) if kind == "pool" else None
    elif kind == "block":
        B, S, d = case["B"], case["S"], case["d"]
        with torch.device(DEV):
            s["layer"] = TransformerBlock(_dense_config(d, case["ff"], case["heads"]))
        _running(s["layer"], g)
        s["x"] = rnd(B, S, d).requires_grad_()
        s["dy"] = rnd(B, S, d)
    elif kind == "swiglu":
        T, d = case["T"], case["d"]
        with torch.device(DEV):
            s["layer"] = DenseSwiGLU(_dense_config(d, case["ff"]))
        s["x"] = rnd(T, d).to(BF16).requires_grad_(bool(case["grad"]))
        s["dy"] = rnd(T, d) if case["grad"] else None
    elif kind == "svd":
        T, d, ff, r = case["T"], case["d"], case["ff"], case["r"]

        def factor(m):  # U or V of a truncated SVD: orthonormal columns
            return torch.linalg.qr(rnd(m, r))[0]

        def values():  # singular values over two decades
            return 10.0 ** (torch.rand(r, device=DEV, generator=g) * 2.0 - 2.0)

        w = [torch.cat([factor(d) * values(), factor(d) * values()], 1), torch.cat([factor(ff), factor(ff)], 0),
             factor(ff), factor(d) * values()]
        s["weights"] = [nn.Parameter(t.contiguous()) for t in w]
        s["x"] = rnd(T, d).to(BF16).requires_grad_()
        s["dy"] = rnd(T, d)
    elif kind == "head":
        T, d, V = case["T"], case["d"], case["V"]
        s["w"] = nn.Parameter(rnd(V, d) * 0.05)
        s["x"] = rnd(T, d).to(BF16).requires_grad_()
        s["targets"] = _zipf((T,), V, g)
        s["dloss"] = torch.full((T,), 1.0 / T, device=DEV)
    else:
        B, S, d, V = case["B"], case["S"], case["d"], case["V"]
        with torch.device(DEV):
            s["head"] = ShortlistHead(d, V, OutputConfig(mode="shortlist"))
        s["w"] = nn.Parameter(rnd(V, d) * 0.05)
        s["x"] = rnd(B, S, d).to(BF16).requires_grad_()
        s["targets"] = _zipf((B, S), V, g)
        s["negatives"] = s["head"].random_negatives(B, S, seed, DEV)
        s["dloss"] = torch.full((B,), 1.0 / (B * S), device=DEV)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "eval":
        with torch.no_grad():
            return s["model"].forward_macro(s["tokens"], fixed_recipe=s["recipe"], fixed_depth=4).logits
    if kind == "step":
        res = s["engine"].train_step((s["tokens"], s["targets"]))
        return {"loss": res.loss, "logits": res.model_output.logits,
                "weights": list(s["engine"].recursive_model.parameters())}
    if kind in ("pool", "pool_eval", "block", "swiglu"):
        layer, x, dy = s["layer"], s["x"], s["dy"]
        if dy is None:
            with torch.no_grad():
                y = layer(x)
            return {"y": y, "ids": layer.last_ids} if kind == "pool_eval" else {"y": y}
        with hip_ops.fp32_precision(bool(case.get("fp32"))):
            y = layer(x)
            grads = torch.autograd.grad(y, [x, *layer.parameters()], dy)
        out = {"y": y, "grads": list(grads)}
        if kind == "pool":
            out["ids"] = layer.last_ids
        return out
    if kind == "svd":
        y = hip_ops.svd_ffn(s["x"], *s["weights"])
        return {"y": y, "grads": list(torch.autograd.grad(y, [s["x"], *s["weights"]], s["dy"]))}
    if kind == "head":
        logits, loss = hip_ops.lm_head_ce(s["x"], s["w"], s["targets"])
        return {"logits": logits, "loss": loss,
                "grads": list(torch.autograd.grad(loss, [s["x"], s["w"]], s["dloss"]))}
    res = s["head"].loss(s["x"], s["targets"], s["w"], seed=0, random_negs=s["negatives"])
    return {"logits": res.logits, "loss": res.loss_per_sample, "shortlist": res.shortlist,
            "grads": list(torch.autograd.grad(res.loss_per_sample, [s["x"], s["w"]], s["dloss"]))}


# ----------------------------------------------------------------------------- work and tolerance

def work(case):
    kind = case["kind"]
    T = case["T"] if "T" in case else case["B"] * case["S"]
    d = case["d"]
    if kind in ("pool", "pool_eval"):
        C, n, k = case["C"], case["n"], case["k"]
        w = 3 * C * n * d + C * d
        fwd = T * k * 6.0 * d * n + 2.0 * T * d * C
        xb = 4 if case.get("fp32") else 2
        if kind == "pool_eval":
            return {"flops": fwd, "bytes": xb * T * d + 4.0 * w + 4.0 * T * d + 4.0 * T * k}
        return {"flops": 3 * fwd, "bytes": 2.0 * xb * T * d + 8.0 * T * d + 8.0 * w + 4.0 * T * k}
    if kind == "block":
        S, ff = case["S"], case["ff"]
        w = 4 * d * d + 3 * d * ff + 2 * d
        return {"flops": 3.0 * T * (2.0 * w + 2.0 * S * d), "bytes": 16.0 * T * d + 8.0 * w}
    if kind == "swiglu":
        w = 3 * d * case["ff"]
        if not case["grad"]:
            return {"flops": 2.0 * T * w, "bytes": 6.0 * T * d + 4.0 * w}
        return {"flops": 6.0 * T * w, "bytes": 12.0 * T * d + 8.0 * w}
    if kind == "svd":
        w = 3 * d * case["r"] + 3 * case["ff"] * case["r"]
        return {"flops": 6.0 * T * w, "bytes": 12.0 * T * d + 8.0 * w}
    if kind == "head":
        V = case["V"]
        return {"flops": 6.0 * T * V * d, "bytes": 4.0 * T * d + 4.0 * T * V + 16.0 * T + 8.0 * V * d}
    if kind == "shortlist":
        L = OutputConfig().shortlist_max_tokens
        return {"flops": 6.0 * T * L * d + 2.0 * T * OutputConfig().num_clusters * d,
                "bytes": 4.0 * T * d + 12.0 * T * L + 8.0 * case["V"] * d}
    # whole model: two blocks with routed pools (top-8 of 64 x 32), router, rank-32 operator, tied head
    mc = _model_config(d)
    V, n, k, C, r = mc.vocab_size, mc.d_ff // mc.ffn_clusters, mc.ffn_top_k, mc.ffn_clusters, mc.macro_rank
    block = 2.0 * 4 * d * d + 2.0 * case["S"] * d + 6.0 * k * n * d + 2.0 * C * d
    macro = 2.0 * (3 * d * r + r * d)
    blockw = 4 * d * d + 3 * C * n * d + C * d + 2 * d
    if kind == "eval":
        return {"flops": T * (2 * block + macro + 2.0 * V * d),
                "bytes": 4.0 * (2 * blockw + V * d + 4 * d * r) + 8.0 * T + 4.0 * T * V}
    # the step: the hot path three times, the consistency term's five operator applications, the
    # audited sequence's four banked passes and its coda and head; every weight and its two moments
    # read and written, every gradient written and read
    hot = 3 * T * (2 * block + 6 * macro + 2.0 * V * d)
    audit = 3 * case["S"] * (4 * (2.0 * d * d + 6.0 * 256 * d) + block + 2.0 * V * d)
    params = 2 * blockw + V * d + 3 * (d * d + d) + (4 * d * d + 3 * mc.d_ff * d) + 48 * (4 * d * r + 2 * d)
    return {"flops": hot + audit, "bytes": 32.0 * params + 4.0 * T * V}


# The relative error of two correct implementations at the same precision.  Every product summed
# in the opposite order within its steps changes the results by at most a quarter of these figures
# in the whole calls (eval 2.6e-4, step 4e-3) and the block (3.6e-3), whose layers' bf16 rounding
# carries on into the next; the single layers change by 3e-4 or less then, and there the line is
# what two different placements of the same bf16 roundings differ by (1.4 times the error against
# `exact`: pool, svd 4e-3, swiglu 3.5e-3, head 2.4e-3, shortlist 1.8e-3).  `max` leaves room for a
# few bf16 steps of one element, in the whole models for a token whose last routed cluster is a tie.
_TOLERANCE = {
    "eval": {"rel": 6e-3, "max": 0.3},
    "pool": {"rel": 6e-3, "max": 0.06, "differ": 1e-3},
    "pool_fp32": {"rel": 1e-5, "max": 1e-3, "differ": 1e-3},
    "pool_eval": {"rel": 6e-3, "max": 0.06, "differ": 1e-3},
    "block": {"rel": 1.4e-2, "max": 0.1},
    "swiglu": {"rel": 6e-3, "max": 0.06},
    "svd": {"rel": 6e-3, "max": 0.06},
    "head": {"rel": 4e-3, "max": 0.06},
    "shortlist": {"rel": 3e-3, "max": 0.06, "differ": 1e-3},
    "step": {"rel": 1.6e-2, "max": 0.5},
}


def tolerance(case):
    return _TOLERANCE["pool_fp32" if case.get("fp32") else case["kind"]]


# ----------------------------------------------------------------------------- 64-bit results

def _leaf(t, bf16=True):
    """t in 64 bits; bf16: its bf16 value, as the path's operands are."""
    t = t.detach()
    return (t.to(BF16) if bf16 else t).to(F64).requires_grad_()


def _swiglu(x, wug, wd):
    up, gate = (x @ wug.t()).chunk(2, dim=-1)
    return (up * F.silu(gate)) @ wd.t()


def _pool(x, wr, wug, wd, k):
    """Top-k routed pools: softmax over the selected logits weights each cluster's SwiGLU."""
    T, C, ff = x.shape[0], wr.shape[0], wd.shape[1]
    n = ff // C
    top, ids = (x @ wr.t()).topk(k, dim=-1)
    w = top.softmax(dim=-1)
    y = torch.zeros_like(x)
    for c in range(C):
        tok, j = (ids == c).nonzero(as_tuple=True)
        if tok.numel():
            own = slice(c * n, (c + 1) * n)
            z = _swiglu(x[tok], torch.cat([wug[own], wug[ff + c * n:ff + (c + 1) * n]]), wd[:, own])
            y = y.index_add(0, tok, w[tok, j].unsqueeze(1) * z)
    return y


def _norm(x, w, eps=1e-5):
    return x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + eps) * w


def _attention(x, wqkv, wo, heads):
    B, S, d = x.shape
    hd = d // heads
    q, k, v = (t.transpose(1, 2) for t in (x @ wqkv.t()).view(B, S, 3, heads, hd).unbind(2))
    freq = 1.0 / (10_000.0 ** (torch.arange(0, hd, 2, device=x.device, dtype=F64) / hd))
    at = torch.outer(torch.arange(S, device=x.device, dtype=F64), freq).repeat_interleave(2, dim=-1)

    def turn(t):
        return t * at.cos() + torch.stack([-t[..., 1::2], t[..., 0::2]], dim=-1).flatten(-2) * at.sin()

    scores = turn(q).contiguous() @ turn(k).transpose(-1, -2).contiguous() / hd**0.5
    later = torch.ones(S, S, dtype=torch.bool, device=x.device).triu(1)
    y = scores.masked_fill(later, float("-inf")).softmax(dim=-1) @ v.contiguous()
    return y.transpose(1, 2).reshape(B, S, d) @ wo.t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return None  # the engine's composed step: its layers are the other cases
    s = prepare(case, seed)
    if kind == "eval":
        return _exact_eval(s)
    if kind in ("pool", "pool_eval"):
        fp32 = bool(case.get("fp32"))
        x = _leaf(s["x"], not fp32)
        w = [_leaf(p, not fp32) for p in s["layer"].parameters()]  # router, wug, wd
        if kind == "pool_eval":
            with torch.no_grad():
                return {"y": _pool(x, *w, case["k"]), "ids": None}
        y = _pool(x, *w, case["k"])
        return {"y": y.detach(), "grads": list(torch.autograd.grad(y, [x, *w], s["dy"].to(F64))), "ids": None}
    if kind == "block":
        p = {k: _leaf(v, v.dim() > 1) for k, v in s["layer"].named_parameters()}
        x = _leaf(s["x"], False)
        y = _exact_block(x, p, case["heads"])
        return {"y": y.detach(), "grads": list(torch.autograd.grad(y, [x, *p.values()], s["dy"].to(F64)))}
    if kind == "swiglu":
        x, w = _leaf(s["x"]), [_leaf(p) for p in s["layer"].parameters()]
        if not case["grad"]:
            with torch.no_grad():
                return {"y": _swiglu(x, *w)}
        y = _swiglu(x, *w)
        return {"y": y.detach(), "grads": list(torch.autograd.grad(y, [x, *w], s["dy"].to(F64)))}
    if kind == "svd":
        x, w = _leaf(s["x"]), [_leaf(p) for p in s["weights"]]
        us_ug, v_ug, v_dn, us_dn = w
        r, ff = case["r"], case["ff"]
        a = x @ us_ug
        z = (a[:, :r] @ v_ug[:ff].t()) * F.silu(a[:, r:] @ v_ug[ff:].t())
        y = (z @ v_dn) @ us_dn.t()
        return {"y": y.detach(), "grads": list(torch.autograd.grad(y, [x, *w], s["dy"].to(F64)))}
    x, w = _leaf(s["x"]), _leaf(s["w"])
    if kind == "head":
        logits = x @ w.t()
        loss = F.cross_entropy(logits, s["targets"], reduction="none")
        return {"logits": logits.detach(), "loss": loss.detach(),
                "grads": list(torch.autograd.grad(loss, [x, w], s["dloss"].to(F64)))}
    return _exact_shortlist(s, x, w)


def _exact_block(x, p, heads):
    y = x + _attention(_norm(x, p["norm1.weight"]), p["attn.wqkv.weight"], p["attn.wo.weight"], heads)
    n = _norm(y, p["norm2.weight"])
    if "mlp.router.weight" not in p:
        return y + _swiglu(n, p["mlp.wug.weight"], p["mlp.wd.weight"])
    flat = n.reshape(-1, n.shape[-1])
    return y + _pool(flat, p["mlp.router.weight"], p["mlp.wug.weight"], p["mlp.wd.weight"], 8).view_as(y)


def _exact_eval(s):
    m = s["model"]
    cfg = m.config

    def params(block):
        return {k: _leaf(v, v.dim() > 1) for k, v in block.named_parameters()}

    with torch.no_grad():
        h = m.embed.weight.detach().to(F64)[s["tokens"]]
        h = _exact_block(h, params(m.prelude[0]), cfg.n_heads)
        o, at = m.macro, (s["recipe"], cfg.depth_choices.index(4))
        z = h * torch.rsqrt(h.pow(2).mean(dim=-1, keepdim=True) + 1e-5)
        z = torch.cat([z, z.mean(dim=1, keepdim=True).expand_as(z), h], dim=-1)
        low = F.silu(z @ _leaf(o.v[at])) @ _leaf(o.u[at])
        push = torch.tanh(o.d_gain[at].to(F64) * h + low + o.bias[at].to(F64))
        h = h + cfg.macro_update_scale * o.update_scale[at].to(F64) * push
        h = _exact_block(h, params(m.coda[0]), cfg.n_heads)
        return _norm(h, m.final_norm.weight.detach().to(F64)) @ _leaf(m.embed.weight).t()


def _exact_shortlist(s, x, w):
    """Candidates in order [target, members of the top clusters, hard, random, fillers], the first
    of each id kept, the first L of those; cross-entropy with the target at position 0."""
    head, targets = s["head"], s["targets"]
    V, cfg = w.shape[0], head.config
    B, S = targets.shape
    T, L = B * S, cfg.shortlist_max_tokens
    flat = x.reshape(T, -1)
    with torch.no_grad():
        top = (flat @ _leaf(head.cluster_router.weight).t()).topk(cfg.shortlist_top_clusters, dim=-1).indices
        t = targets.reshape(T, 1)
        fill = torch.arange(max(2 * L, cfg.hard_negatives), device=x.device)

        def same(ids):
            return (ids % V).expand(T, -1)

        ids = torch.cat([t, head.cluster_members[top].reshape(T, -1), same(fill[:cfg.hard_negatives]),
                         s["negatives"].reshape(T, -1), same(fill[:L]), (t + fill[:2 * L]) % V], dim=1)
        order = ids.sort(dim=1, stable=True)
        new = torch.ones_like(ids, dtype=torch.bool)
        new[:, 1:] = order.values[:, 1:] != order.values[:, :-1]
        first = torch.zeros_like(new).scatter(1, order.indices, new)
        place = torch.where(first, torch.arange(ids.shape[1], device=x.device), ids.shape[1])
        keep = place.topk(L, dim=1, largest=False, sorted=True).indices
        sl = ids.gather(1, keep)
    logits = (flat @ w.t()).gather(1, sl)
    loss = (torch.logsumexp(logits, dim=-1) - logits[:, 0]).view(B, S).sum(dim=-1)
    grads = torch.autograd.grad(loss, [x, w], s["dloss"].to(F64))
    return {"logits": logits.detach().view(B, S, L), "loss": loss.detach(), "shortlist": None, "grads": list(grads)}
