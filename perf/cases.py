"""The work a user of this framework has it do, as measurable cases.

Each case runs one pass of a public entry point, forward and backward, on
inputs made on the GPU from a seed:

  stream   the bandwidth-bound operators of the headline benchmark: RMSNorm and
           SwiGLU, forward and backward (the registered operators)
  addnorm  the residual add with the RMSNorm that reads it, forward and
           backward (FusedAddRMSNorm), as every block runs it
  mlp      the token-tiled SwiGLU MLP under fp16 autocast (TiledMLP)
  attn     the causal attention layer under fp16 autocast: qkv projection,
           attention, output projection (enable_linear, enable_attention)
  head     the tied LM head with its cross-entropy (tied_head_ce)
  optim    gradient unscale and clip, then AdamW (FusedAdamW)
  step     one training step of a reversible decoder (cached_head_backward on
           an install_v3 model), captured once and replayed (CapturedStep)

With "graph" an mlp or attn pass is captured and replayed as well, as inside a
captured training step; without it every launch is made from Python.

Sizes are the decoder configurations this repository trains and benchmarks
(width 256, 7 layers, 512 tokens; width 1024, 12 layers, 2048 tokens), the
small and odd shapes of its tests, and the ranges between them.
"""
import math

import torch
import torch.nn.functional as F

from reversability_amd import ModelConfig, build_model
from reversability_amd._hip import ops
from reversability_amd.attention import enable_attention
from reversability_amd.embedding import enable_embedding
from reversability_amd.graph import CapturedStep
from reversability_amd.kernels import padded_head, tied_head_ce
from reversability_amd.kernels_v3 import FusedAddRMSNorm
from reversability_amd.linear import enable_linear
from reversability_amd.model import BaselineLM
from reversability_amd.optim import FusedAdamW
from reversability_amd.optimized_v3 import TiledMLP, cached_head_backward, install_v3

EPS = float(torch.finfo(torch.float32).eps)
VOCAB = 50257
SCALE = 65536.0  # GradScaler's initial scale
DTYPES = {"fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # the headline benchmark: both operators at 29 sequences of 512 tokens
        {"name": "stream_29x512", "kind": "stream", "rows": 29 * 512, "width": 256,
         "hidden": 1024, "dtype": "fp16"},
        # the wide decoder's residual add + norm, 16 sequences of 2048 tokens
        {"name": "addnorm_16x2048", "kind": "addnorm", "rows": 16 * 2048, "width": 1024,
         "force": "fp16"},
        # the smallest MLP call: 3 sequences of 17 tokens, all latency and launches
        {"name": "mlp_3x17", "kind": "mlp", "rows": 51, "d": 256, "f": 1024, "tile": 8192,
         "keep": False, "x": "fp32", "graph": False},
        # the MLP block benchmark: 8192-token tiles, recomputed in the backward
        {"name": "mlp_29x512", "kind": "mlp", "rows": 29 * 512, "d": 256, "f": 1024,
         "tile": 8192, "keep": False, "x": "fp32", "graph": True},
        # the wide decoder's MLP on a few odd-length sequences
        {"name": "mlp_2x1531", "kind": "mlp", "rows": 2 * 1531, "d": 1024, "f": 4096,
         "tile": 32768, "keep": True, "x": "fp16", "graph": False},
        # the wide decoder's MLP inside its training step: one tile, tiles kept
        {"name": "mlp_16x2048", "kind": "mlp", "rows": 16 * 2048, "d": 1024, "f": 4096,
         "tile": 32768, "keep": True, "x": "fp16", "graph": False},
        # the narrow decoder's attention layer (head size 32)
        {"name": "attn_33x512", "kind": "attn", "batch": 33, "seq": 512, "heads": 8, "hd": 32,
         "graph": True},
        # the wide decoder's attention layer (head size 64)
        {"name": "attn_16x2048", "kind": "attn", "batch": 16, "seq": 2048, "heads": 16, "hd": 64,
         "graph": False},
        # a few ragged sequences at the largest head size
        {"name": "attn_3x777", "kind": "attn", "batch": 3, "seq": 777, "heads": 4, "hd": 128,
         "graph": False},
        # the narrow decoder's tied head over its whole batch
        {"name": "head_33x512", "kind": "head", "rows": 33 * 512, "d": 256, "vocab": VOCAB},
        # the optimizer over three layers of the wide decoder and its embeddings
        {"name": "optim_3L1024", "kind": "optim", "layers": 3, "d": 1024, "f": 4096,
         "vocab": VOCAB, "seq": 2048},
        # the narrow decoder's whole training step
        {"name": "step_33x512", "kind": "step", "method": "midpoint", "layers": 7, "batch": 33,
         "seq": 512, "heads": 8, "hd": 32, "vocab": VOCAB},
    ]


def _log(rng, low, high):
    """An integer spread over the logarithm of [low, high]."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["stream", "addnorm", "mlp", "mlp", "attn", "attn", "head", "optim", "step"])
    if kind == "stream":
        rows = _log(rng, 64, 29 * 512)
        if rng.random() < 0.5:
            width, hidden = 8 * rng.randint(8, 128), 8 * rng.randint(16, 256)
        else:  # any width
            width, hidden = rng.randint(64, 1024), rng.randint(128, 2048)
        return {"kind": kind, "rows": rows, "width": width, "hidden": hidden,
                "dtype": rng.choice(["fp16", "fp16", "fp32"])}
    if kind == "addnorm":
        width = 4 * rng.randint(32, 512)
        return {"kind": kind, "rows": _log(rng, 64, 2 ** 25 // width), "width": width,
                "force": rng.choice(["fp16", "fp16", "fp32"])}
    if kind == "mlp":
        d = 128 * rng.randint(1, 8)
        f = 128 * rng.randint(2, 32)
        rows = _log(rng, 17, min(32768, 32768 * 1024 * 4096 // (d * f)))
        return {"kind": kind, "rows": rows, "d": d, "f": f, "tile": rng.choice([8192, 32768]),
                "keep": rng.random() < 0.5, "x": rng.choice(["fp16", "fp32"]),
                "graph": rng.random() < 0.5}
    if kind == "attn":
        hd = rng.choice([32, 64, 128])
        heads = {32: 4, 64: 2, 128: 1}[hd] * rng.randint(1, 8)
        seq = _log(rng, 17, 2048)
        return {"kind": kind, "batch": _log(rng, 1, max(1, 16 * 2048 // seq)), "seq": seq,
                "heads": heads, "hd": hd, "graph": rng.random() < 0.5}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 64, 33 * 512), "d": rng.choice([128, 256]),
                "vocab": _log(rng, 1000, VOCAB)}
    if kind == "optim":
        d = 64 * rng.randint(2, 16)
        return {"kind": kind, "layers": rng.randint(1, 3), "d": d, "f": rng.choice([3, 4]) * d,
                "vocab": _log(rng, 1000, VOCAB), "seq": rng.choice([512, 1024, 2048])}
    hd = rng.choice([32, 64])
    return {"kind": kind, "method": rng.choice(["midpoint", "euler"]), "layers": rng.randint(1, 6),
            "batch": rng.randint(1, 33), "seq": rng.randint(64, 512),
            "heads": 256 // hd, "hd": hd, "vocab": _log(rng, 1000, VOCAB)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda").mul_(std).to(dtype)


def _decoder(case):
    """A reversible decoder wired as the training step runs it."""
    d = case["heads"] * case["hd"]
    with torch.device("cuda"):
        model = build_model({"model": {"vocab_size": case["vocab"],
                                       "max_sequence_length": case["seq"],
                                       "n_layers": case["layers"], "n_heads": case["heads"],
                                       "d_model": d, "d_ff": 4 * d}, "method": case["method"]})
    return model


def _reseed(model, g):
    """Weights of the decoder's own initialisation, from ``g``, norm weights near one."""
    with torch.no_grad():
        for name, p in model.named_parameters():
            if p.ndim == 1:
                p.copy_(1 + 0.02 * torch.randn(p.shape, generator=g, device="cuda"))
            else:
                residual = name.endswith(("attn.proj.weight", "mlp.down.weight"))
                std = 0.02 / math.sqrt(2 * model.config.n_layers) if residual else 0.02
                p.copy_(std * torch.randn(p.shape, generator=g, device="cuda"))


def _inputs(case, seed):
    """The seeded tensors of a case, without this framework's wiring."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "stream":
        rows, w, h, t = case["rows"], case["width"], case["hidden"], DTYPES[case["dtype"]]
        return {"x": _randn(g, rows, w), "w": 1 + _randn(g, w, std=0.02), "dy": _randn(g, rows, w),
                "u": _randn(g, rows, 2 * h, dtype=t), "do": _randn(g, rows, h, dtype=t)}
    if kind == "addnorm":
        rows, w = case["rows"], case["width"]
        return {"x": _randn(g, rows, w), "f": _randn(g, rows, w, std=0.3,
                                                     dtype=DTYPES[case["force"]]),
                "w": 1 + _randn(g, w, std=0.02), "dh": _randn(g, rows, w),
                "dy": _randn(g, rows, w, dtype=torch.float16)}
    if kind == "mlp":
        rows, d, f = case["rows"], case["d"], case["f"]
        return {"x": _randn(g, rows, d, dtype=DTYPES[case["x"]]), "up": _randn(g, 2 * f, d, std=0.02),
                "down": _randn(g, d, f, std=0.02 / math.sqrt(14)),
                "dy": _randn(g, rows, d, dtype=torch.float16)}
    if kind == "attn":
        d = case["heads"] * case["hd"]
        shape = (case["batch"], case["seq"], d)
        return {"x": _randn(g, *shape, dtype=torch.float16), "qkv": _randn(g, 3 * d, d, std=0.05),
                "proj": _randn(g, d, d, std=0.02), "dy": _randn(g, *shape, dtype=torch.float16)}
    if kind == "head":
        rows, d, vocab = case["rows"], case["d"], case["vocab"]
        labels = torch.randint(0, vocab, (rows,), generator=g, device="cuda")
        labels[torch.rand(rows, generator=g, device="cuda") < 0.02] = -100
        return {"x": _randn(g, rows, d, dtype=torch.float16), "w": _randn(g, vocab, d, std=0.02),
                "labels": labels, "grad": torch.full((1,), SCALE / rows, device="cuda")}
    if kind == "optim":
        d, f = case["d"], case["f"]
        shapes = [(case["vocab"], d), (case["seq"], d)]
        for _ in range(case["layers"]):
            shapes += [(d,), (3 * d, d), (d, d), (d,), (2 * f, d), (d, f)]
        shapes.append((d,))
        return {"params": [_randn(g, *s, std=0.02) for s in shapes],
                "grads": [_randn(g, *s, std=0.05) for s in shapes]}
    tokens = torch.randint(0, case["vocab"], (case["batch"], case["seq"] + 1), generator=g,
                           device="cuda")
    return {"ids": tokens[:, :-1].contiguous(), "labels": tokens[:, 1:].contiguous(), "gen": g}


def prepare(case, seed):
    kind = case["kind"]
    state = _inputs(case, seed)
    state["kind"] = kind
    if kind == "addnorm":
        for k in ("x", "f", "w"):
            state[k].requires_grad_(True)
    elif kind == "mlp":
        for k in ("x", "up", "down"):
            state[k].requires_grad_(True)
        state["tile"], state["keep"] = case["tile"], case["keep"]
    elif kind == "attn":
        d = case["heads"] * case["hd"]
        with torch.device("cuda"):
            model = BaselineLM(ModelConfig(vocab_size=64, max_sequence_length=case["seq"],
                                           n_layers=1, n_heads=case["heads"], d_model=d,
                                           d_ff=d))
        enable_linear(model)
        enable_attention(model)
        attn = model.blocks[0].attn
        with torch.no_grad():
            attn.qkv.weight.copy_(state.pop("qkv"))
            attn.proj.weight.copy_(state.pop("proj"))
        state["x"].requires_grad_(True)
        state["attn"] = attn
    elif kind == "head":
        state["head"] = padded_head(state.pop("w"))
        state["vocab"] = case["vocab"]
    elif kind == "optim":
        params = [torch.nn.Parameter(p) for p in state.pop("params")]
        for p, grad in zip(params, state.pop("grads")):
            p.grad = grad
        state["params"] = params
        state["opt"] = FusedAdamW(params, lr=6e-4, betas=(0.9, 0.95), weight_decay=0.1)
    elif kind == "step":
        model = _decoder(case)
        _reseed(model, state.pop("gen"))
        targets = case["batch"] * case["seq"]
        install_v3(model, core_mode="split" if case["method"] == "midpoint" else "reference",
                   mlp_tokens=targets, swiglu=True, rmsnorm=True, keep_mlp_tiles=True)
        enable_linear(model)
        enable_attention(model)
        enable_embedding(model, into_grad=True)
        scaler = torch.amp.GradScaler("cuda", init_scale=SCALE)
        ids, labels = state["ids"], state["labels"]

        def step():
            model.zero_grad(set_to_none=True)
            return cached_head_backward(model, ids, labels, targets, targets, scaler, "fp16",
                                        False, "hip")

        state["model"], state["step"] = model, CapturedStep(step)
    if case.get("graph"):
        state["step"] = CapturedStep(lambda s=dict(state): _eager(s))
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    if "step" not in state:
        return _eager(state)
    out = state["step"]()
    if state["kind"] == "step":
        return {"loss": out, "grads": [p.grad for p in state["model"].parameters()]}
    return out


def _eager(state):
    kind = state["kind"]
    if kind == "stream":
        y, rstd = ops.rmsnorm_fwd(state["x"], state["w"], EPS)
        o = ops.swiglu_fwd(state["u"])
        du = ops.swiglu_bwd(state["u"], state["do"])
        dx, dw = ops.rmsnorm_bwd(state["x"], state["w"], state["dy"], rstd)
        return {"y": y, "o": o, "du": du, "dx": dx, "dw": dw}
    if kind == "addnorm":
        leaves = (state["x"], state["f"], state["w"])
        with torch.autocast("cuda", dtype=torch.float16):
            h, y = FusedAddRMSNorm.apply(*leaves, EPS)
        dx, df, dw = torch.autograd.grad((h, y), leaves, (state["dh"], state["dy"]))
        return {"h": h.detach(), "y": y.detach(), "dx": dx, "df": df, "dw": dw}
    if kind == "mlp":
        leaves = (state["x"], state["up"], state["down"])
        with torch.autocast("cuda", dtype=torch.float16):
            y = TiledMLP.apply(*leaves, state["tile"], True, state["keep"])
        dx, dup, ddown = torch.autograd.grad(y, leaves, state["dy"])
        return {"y": y.detach(), "dx": dx, "dup": dup, "ddown": ddown}
    if kind == "attn":
        attn = state["attn"]
        with torch.autocast("cuda", dtype=torch.float16):
            y = attn(state["x"])
        dx, dqkv, dproj = torch.autograd.grad(y, (state["x"], attn.qkv.weight, attn.proj.weight),
                                              state["dy"])
        return {"y": y.detach(), "dx": dx, "dqkv": dqkv, "dproj": dproj}
    if kind == "head":
        loss, dx, dw = tied_head_ce(state["x"], state["head"], state["vocab"], state["labels"],
                                    state["grad"])
        return {"loss": loss, "dx": dx, "dw": dw}
    opt = state["opt"]
    norm = opt.unscale_clip_(None, 1.0)
    opt.step()
    return {"norm": norm, "params": [p.detach() for p in state["params"]],
            "m": [opt.state[p]["exp_avg"] for p in state["params"]],
            "v": [opt.state[p]["exp_avg_sq"] for p in state["params"]]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "stream":
        rows, w, h = case["rows"], case["width"], case["hidden"]
        size = 2 if case["dtype"] == "fp16" else 4
        # x twice (it outlives no pass), dy, y, dx; u twice, do, o, du
        return {"bytes": rows * w * 4 * 5 + rows * h * size * 8,
                "flops": rows * w * 14 + rows * h * 20}
    if kind == "addnorm":
        rows, w, f = case["rows"], case["width"], 2 if case["force"] == "fp16" else 4
        # forward x, f, h, y; backward h, dh, dy, dx, df
        return {"bytes": rows * w * (4 + f + 4 + 2 + 4 + 4 + 2 + 4 + f), "flops": rows * w * 18}
    if kind == "mlp":
        rows, d, f = case["rows"], case["d"], case["f"]
        x = 2 if case["x"] == "fp16" else 4
        return {"bytes": rows * d * (2 * x + 2 + 2) + 3 * f * d * 4 * 2,
                "flops": 18 * rows * d * f}
    if kind == "attn":
        b, t, d = case["batch"], case["seq"], case["heads"] * case["hd"]
        rows = b * t
        # projections 3 x 2 x 4 d^2 per token, attention 4 + 10 per visible pair and column
        return {"bytes": rows * d * 2 * 4 + 4 * d * d * 4 * 2,
                "flops": 24 * rows * d * d + 14 * b * d * t * (t + 1) // 2}
    if kind == "head":
        rows, d, vocab = case["rows"], case["d"], case["vocab"]
        return {"bytes": (2 * rows * d + 2 * vocab * d) * 2 + rows * 8,
                "flops": 6 * rows * d * vocab}
    if kind == "optim":
        d, f = case["d"], case["f"]
        n = (case["vocab"] + case["seq"]) * d + d
        n += case["layers"] * (2 * d + 4 * d * d + 3 * d * f)
        return {"bytes": 28 * n, "flops": 16 * n}
    d, t = case["heads"] * case["hd"], case["seq"]
    rows = case["batch"] * t
    matrix = case["layers"] * 16 * d * d
    n = matrix + case["layers"] * 2 * d + (case["vocab"] + t + 1) * d
    return {"bytes": 8 * n + 16 * rows,
            "flops": 6 * rows * (matrix + case["vocab"] * d)
            + 14 * case["layers"] * case["batch"] * d * t * (t + 1) // 2}


def tolerance(case):
    """About four times the largest relative difference from ``exact`` that the
    listed and some drawn cases show."""
    kind = case["kind"]
    if kind == "stream":  # fp32 sums; SwiGLU rounds to its input type
        return {"rel": 1e-3 if case["dtype"] == "fp16" else 1e-5}
    if kind == "addnorm":
        return {"rel": 1e-3}
    # fp16 operands and results, fp32 sums
    if kind == "mlp":
        return {"rel": 2.6e-3}
    if kind == "attn":
        return {"rel": 4e-3}
    if kind == "head":
        return {"rel": 1.2e-3}
    if kind == "optim":
        return {"rel": 1e-5}
    return {"rel": 8e-3}  # fp16 through every layer and its reconstruction


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _grads(out, leaves, cotangents):
    return torch.autograd.grad(out, leaves, cotangents)


def _leaf(t):
    return t.detach().double().requires_grad_(True)


def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _swiglu64(u):
    gate, value = u.chunk(2, -1)
    return F.silu(gate) * value


def _attention64(qkv, heads):
    """Causal attention of a packed [B, T, 3 d] projection."""
    b, t, width = qkv.shape
    d = width // 3
    q, k, v = qkv.view(b, t, 3, heads, d // heads).permute(2, 0, 3, 1, 4).unbind(0)
    return _sdpa64(q, k, v).transpose(1, 2).reshape(b, t, d)


def _sdpa64(q, k, v):
    t = q.shape[-2]
    hidden = torch.ones(t, t, dtype=torch.bool, device=q.device).triu(1)
    scores = q.contiguous() @ k.transpose(-1, -2).contiguous() / math.sqrt(q.shape[-1])
    return scores.masked_fill(hidden, -math.inf).softmax(-1) @ v.contiguous()


def _head64(x, w, labels, grad):
    """Summed cross-entropy of x w^T and its gradients at upstream gradient ``grad``."""
    loss, dx, dw = 0.0, torch.empty_like(x), torch.zeros_like(w)
    for at in range(0, x.shape[0], 2048):
        xs, ls = x[at:at + 2048], labels[at:at + 2048]
        logp = (xs @ w.t()).log_softmax(-1)
        loss = loss + F.nll_loss(logp, ls, ignore_index=-100, reduction="sum")
        dl = logp.exp()
        valid = ls >= 0
        dl[valid.nonzero()[:, 0], ls[valid]] -= 1
        dl *= (valid * grad).unsqueeze(1)
        dx[at:at + 2048] = dl @ w
        dw += dl.t() @ xs
    return loss, dx, dw


def _attn64(block, x, heads):
    qkv = _norm64(x, block["attn_norm"]) @ block["qkv"].t()
    return _attention64(qkv, heads) @ block["proj"].t()


def _mlp64(block, x):
    return _swiglu64(_norm64(x, block["mlp_norm"]) @ block["up"].t()) @ block["down"].t()


def _step64(case, seed):
    state = _inputs(case, seed)
    model = _decoder(case)
    _reseed(model, state.pop("gen"))
    params = [_leaf(p) for p in model.parameters()]
    by = dict(zip((n for n, _ in model.named_parameters()), params))
    heads, h = case["heads"], 0.5
    blocks = [{"attn_norm": by[f"blocks.{i}.attn_norm.weight"],
               "mlp_norm": by[f"blocks.{i}.mlp_norm.weight"],
               "qkv": by[f"blocks.{i}.attn.qkv.weight"],
               "proj": by[f"blocks.{i}.attn.proj.weight"],
               "up": by[f"blocks.{i}.mlp.up.weight"],
               "down": by[f"blocks.{i}.mlp.down.weight"]} for i in range(case["layers"])]
    ids, labels = state["ids"], state["labels"]
    p = q = by["token_embedding.weight"][ids] + by["position_embedding.weight"][:case["seq"]]
    for block in blocks:
        if case["method"] == "midpoint":
            a = _attn64(block, q, heads)
            p, q = q, p + 2 * h * (a + _mlp64(block, q + a))
        else:
            q = q + _attn64(block, p, heads)
            p = p + _mlp64(block, q)
    hidden = _norm64(q if case["method"] == "midpoint" else p, by["final_norm.weight"])
    flat = hidden.reshape(-1, hidden.shape[-1])
    head = by["token_embedding.weight"]
    loss, dx, dw = _head64(flat.detach(), head.detach(), labels.reshape(-1),
                           SCALE / labels.numel())
    grads = list(torch.autograd.grad(flat, params, dx))
    at = next(i for i, w in enumerate(params) if w is head)
    grads[at] = grads[at] + dw
    return {"loss": loss, "grads": grads}


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _step64(case, seed)
    s = _inputs(case, seed)
    if kind == "stream":
        x, w, u = _leaf(s["x"]), _leaf(s["w"]), _leaf(s["u"])
        y, o = _norm64(x, w), _swiglu64(u)
        dx, dw, du = _grads((y, o), (x, w, u), (s["dy"].double(), s["do"].double()))
        return {"y": y.detach(), "o": o.detach(), "du": du, "dx": dx, "dw": dw}
    if kind == "addnorm":
        x, f, w = _leaf(s["x"]), _leaf(s["f"]), _leaf(s["w"])
        h = x + f
        y = _norm64(h, w)
        dx, df, dw = _grads((h, y), (x, f, w), (s["dh"].double(), s["dy"].double()))
        return {"h": h.detach(), "y": y.detach(), "dx": dx, "df": df, "dw": dw}
    if kind == "mlp":
        x, up, down = _leaf(s["x"]), _leaf(s["up"]), _leaf(s["down"])
        y = _swiglu64(x @ up.t()) @ down.t()
        dx, dup, ddown = _grads(y, (x, up, down), s["dy"].double())
        return {"y": y.detach(), "dx": dx, "dup": dup, "ddown": ddown}
    if kind == "attn":
        x, wqkv, wproj = _leaf(s["x"]), _leaf(s["qkv"]), _leaf(s["proj"])
        mixed, dqkv = [], []
        qkv = (x @ wqkv.t()).detach()
        dmixed = s["dy"].double() @ wproj.detach()
        for b in range(qkv.shape[0]):  # a sequence at a time: the scores in 64 bits are large
            one = qkv[b:b + 1].requires_grad_(True)
            out = _attention64(one, case["heads"])
            dqkv.append(torch.autograd.grad(out, one, dmixed[b:b + 1])[0])
            mixed.append(out.detach())
        mixed, dqkv = torch.cat(mixed).flatten(0, 1), torch.cat(dqkv).flatten(0, 1)
        flat, dy = x.detach().flatten(0, 1), s["dy"].double().flatten(0, 1)
        return {"y": (mixed @ wproj.detach().t()).reshape(x.shape),
                "dx": (dqkv @ wqkv.detach()).reshape(x.shape),
                "dqkv": dqkv.t() @ flat, "dproj": dy.t() @ mixed}
    if kind == "head":
        w = s["w"].half().double()
        loss, dx, dw = _head64(s["x"].double(), w, s["labels"], s["grad"].double())
        return {"loss": loss, "dx": dx, "dw": dw}
    # one AdamW step from zero moments, the gradients clipped to norm 1
    grads = [t.double() for t in s["grads"]]
    norm = torch.sqrt(sum((t * t).sum() for t in grads))
    coef = min(1.0, 1.0 / (float(norm) + 1e-6))
    params, m, v = [], [], []
    for p, t in zip(s["params"], grads):
        t = t * coef
        m.append(0.1 * t)
        v.append(0.05 * t * t)
        update = (m[-1] / 0.1) / ((v[-1] / 0.05).sqrt() + 1e-8)
        params.append(p.double() * (1 - 6e-4 * 0.1) - 6e-4 * update)
    return {"norm": norm, "params": params, "m": m, "v": v}
