"""Performance cases of the elementwise + loss path, through the aten ops that
a program on the ``supa`` device calls.

Each case is one step of ordinary use: the calls of a model's block or of its
loss and optimizer, forward and, where training runs it, backward.  The sizes
are those of ``bench.py`` and of the tests, and generic ones around them;
``draw`` spreads them over the same ranges.

``prepare`` draws the inputs on the GPU with torch's own seeded generator and
copies them into supa buffers; ``exact`` evaluates the same formulas on the
same inputs in float64 with torch alone.
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "torch-supa_amd"))
import torch_supa  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}
ACTS = {
    "gelu_tanh": lambda v: F.gelu(v, approximate="tanh"),
    "gelu": F.gelu,
    "silu": F.silu,
    "relu": F.relu,
}
IGNORE = -100


def listed():
    return [
        # one token's hidden state through a bias and an activation: serving,
        # two launches on a few KiB
        dict(name="bias_act_token", op="bias_act", rows=1, cols=4096, x="bf16", bias="bf16", act="gelu_tanh",
             layout="dense", train=False),
        # the same pair in training, a batch of 8192 tokens of width 4096,
        # with the activation's gradient and the bias gradient (a sum over tokens)
        dict(name="bias_act_train", op="bias_act", rows=8192, cols=4096, x="bf16", bias="bf16", act="gelu_tanh",
             layout="dense", train=True),
        # float32 training on a width that is no multiple of anything
        dict(name="bias_act_ragged", op="bias_act", rows=6007, cols=2047, x="f32", bias="f32", act="silu",
             layout="dense", train=True),
        # the benchmark's elementwise step at its full size, bf16 + f32 -> f32
        dict(name="bias_act_large", op="bias_act", rows=131072, cols=4096, x="bf16", bias="f32", act="gelu_tanh",
             layout="dense", train=False),
        # the gated activation of a feed-forward block: both halves of one
        # projection, forward and backward
        dict(name="gated_train", op="gated", rows=4096, cols=11008, x="bf16"),
        # the benchmark's language-model loss (bf16 logits, 5 % ignored targets)
        dict(name="lm_loss", op="cross_entropy", rows=8192, cols=128256, x="bf16", ignored=0.05, reduction="mean"),
        # the same loss over a vocabulary of odd size
        dict(name="lm_loss_ragged", op="cross_entropy", rows=4096, cols=50257, x="bf16", ignored=0.05,
             reduction="mean"),
        # per-pixel classification: classes in dim 1, class weights, ignored borders
        dict(name="pixel_loss", op="pixel_loss", batch=8, cols=19, height=512, width=512, x="f32", weighted=True),
        # attention weights of a causal layer, forward and backward
        dict(name="attention_weights", op="attention", batch=4, heads=16, rows=1024, cols=1024, x="bf16"),
        # a normalisation layer written with var_mean, forward and backward
        dict(name="norm_train", op="norm", rows=8192, cols=4096, inner=1, x="f32"),
        # multi-label classification: BCE with a weight per label
        dict(name="multilabel_loss", op="pointwise_loss", kind="bce", rows=4096, cols=8193, x="f32", reduction="mean"),
        # gradient clipping and the fused AdamW step of two blocks' 18 tensors
        dict(name="optimizer_step", op="optimizer", layers=2, width=2048, hidden=5504, fused=True),
    ]


def _log(rng, lo, hi, odd=0.4):
    """A size from [lo, hi], uniform in its logarithm: of odd value for a
    share `odd` of the draws, else a multiple of 8 (where hi allows)."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < odd:
        n |= 1
    elif n >= 16:
        n -= n % 8
    return max(lo, min(hi, n))


def draw(rng):
    op = rng.choice(["bias_act", "bias_act", "gated", "cross_entropy", "cross_entropy", "pixel_loss", "attention",
                     "norm", "norm", "pointwise_loss", "optimizer", "evaluate"])
    x = rng.choice(["f32", "bf16", "bf16", "f16"])
    if op == "bias_act":
        cols = _log(rng, 256, 16384)
        train = rng.random() < 0.6  # training sees batches of tokens, serving single ones too
        rows = _log(rng, 256 if train else 1, min(131072, (1 << 26) // cols))
        return dict(op=op, rows=rows, cols=cols, x=x, bias=rng.choice([x, "f32"]), act=rng.choice(sorted(ACTS)),
                    layout=rng.choice(["dense", "dense", "transposed"]), train=train)
    if op == "gated":
        cols = _log(rng, 256, 16384)
        return dict(op=op, rows=_log(rng, 256, (1 << 26) // cols), cols=cols, x=x)
    if op == "cross_entropy":
        cols = _log(rng, 10, 160000)
        rows = _log(rng, 256, min(32768, (1 << 28) // cols))
        return dict(op=op, rows=rows, cols=cols, x=rng.choice(["bf16", "f32", "f16"]),
                    ignored=rng.choice([0.0, 0.05, 0.3]), reduction=rng.choice(["mean", "mean", "sum", "none"]))
    if op == "pixel_loss":
        cols = _log(rng, 2, 150)
        height, width = _log(rng, 33, 512), _log(rng, 33, 512)
        batch = _log(rng, 1, max(1, min(16, (1 << 26) // (cols * height * width))), odd=1.0)
        return dict(op=op, batch=batch, cols=cols, height=height, width=width, x=rng.choice(["f32", "f32", "bf16"]),
                    weighted=rng.random() < 0.5)
    if op == "attention":
        rows = _log(rng, 64, 2048)
        heads = rng.choice([8, 12, 16, 32])
        return dict(op=op, batch=_log(rng, 1, max(1, min(16, (1 << 26) // (heads * rows * rows))), odd=1.0),
                    heads=heads, rows=rows, cols=rows, x=x)
    if op == "norm":
        if rng.random() < 0.3:  # per channel of an image batch: the statistics run over dims 0 and 2
            cols, inner = _log(rng, 16, 512), _log(rng, 49, 12544)
            return dict(op=op, rows=_log(rng, 2, max(2, min(128, (1 << 25) // (cols * inner)))), cols=cols,
                        inner=inner, x="f32")
        cols = _log(rng, 128, 16384)
        return dict(op=op, rows=_log(rng, 256, (1 << 25) // cols), cols=cols, inner=1, x=x)
    if op == "pointwise_loss":
        cols = _log(rng, 8, 1048576)
        return dict(op=op, kind=rng.choice(["mse", "smooth_l1", "huber", "bce"]), rows=_log(rng, 16, (1 << 25) // cols),
                    cols=cols, x=rng.choice(["f32", "f32", "bf16"]), reduction=rng.choice(["mean", "sum", "none"]))
    if op == "optimizer":
        width = _log(rng, 128, 2048, odd=0.2)
        return dict(op=op, layers=rng.choice([1, 2]), width=width, hidden=width * 11 // 4, fused=rng.random() < 0.7)
    cols = _log(rng, 10, 50000)
    return dict(op="evaluate", rows=_log(rng, 256, min(32768, (1 << 27) // cols)), cols=cols, x=x)


# ------------------------------------------------------------------ inputs
def _randn(g, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(DTYPES[dtype])


def _targets(g, shape, classes, ignored):
    t = torch.randint(0, classes, shape, generator=g, device="cuda")
    if ignored:
        t[torch.rand(shape, generator=g, device="cuda") < ignored] = IGNORE
    return t


def _optimizer_shapes(case):
    w, h = case["width"], case["hidden"]
    return ([(w, w)] * 4 + [(h, w)] * 2 + [(w, h)] + [(w,)] * 2) * case["layers"]


def _inputs(case, seed):
    """The case's inputs on torch's own HIP device, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    op = case["op"]
    if op == "bias_act":
        r, c = case["rows"], case["cols"]
        shape = (c, r) if case["layout"] == "transposed" else (r, c)
        d = dict(x=_randn(g, shape, case["x"]), bias=_randn(g, (c,), case["bias"], 0.02))
        if case["train"]:
            out = "f32" if "f32" in (case["x"], case["bias"]) else case["x"]
            d["gy"] = _randn(g, shape, out)
        return d
    if op == "gated":
        r, c = case["rows"], case["cols"]
        return dict(x=_randn(g, (r, 2 * c), case["x"]), gy=_randn(g, (r, c), case["x"]))
    if op == "cross_entropy":
        r, c = case["rows"], case["cols"]
        d = dict(x=_randn(g, (r, c), case["x"], 2.0), t=_targets(g, (r,), c, case["ignored"]))
        if case["reduction"] == "none":
            d["gy"] = _randn(g, (r,), case["x"])
        return d
    if op == "pixel_loss":
        b, c, h, w = case["batch"], case["cols"], case["height"], case["width"]
        d = dict(x=_randn(g, (b, c, h, w), case["x"], 2.0), t=_targets(g, (b, h, w), c, 0.05))
        if case["weighted"]:
            d["weight"] = (torch.rand(c, generator=g, device="cuda") + 0.5).to(DTYPES[case["x"]])
        return d
    if op == "attention":
        shape = (case["batch"], case["heads"], case["rows"], case["cols"])
        return dict(x=_randn(g, shape, case["x"]), gy=_randn(g, shape, case["x"]),
                    mask=torch.ones(case["rows"], case["cols"], dtype=torch.bool, device="cuda").triu(1))
    if op == "norm":
        r, c, s = case["rows"], case["cols"], case["inner"]
        shape, ws = ((r, c), (c,)) if s == 1 else ((r, c, s), (c, 1))
        return dict(x=_randn(g, shape, case["x"]), w=1 + _randn(g, ws, case["x"], 0.1),
                    b=_randn(g, ws, case["x"], 0.1), gy=_randn(g, shape, case["x"]))
    if op == "pointwise_loss":
        shape = (case["rows"], case["cols"])
        d = dict(x=_randn(g, shape, case["x"]))
        if case["kind"] == "bce":
            d["t"] = (torch.rand(shape, generator=g, device="cuda") < 0.3).to(DTYPES[case["x"]])
            d["pw"] = (torch.rand(shape[1], generator=g, device="cuda") * 1.5 + 0.5).to(DTYPES[case["x"]])
        else:
            d["t"] = _randn(g, shape, case["x"])
        if case["reduction"] == "none":
            d["gy"] = _randn(g, shape, case["x"])
        return d
    if op == "optimizer":
        d = {}
        for i, s in enumerate(_optimizer_shapes(case)):
            d["p%d" % i] = _randn(g, s, "f32", 0.02)
            d["g%d" % i] = _randn(g, s, "f32", 1e-3)
            d["m%d" % i] = _randn(g, s, "f32", 1e-4)
            d["v%d" % i] = torch.rand(s, generator=g, device="cuda") * 1e-6
        return d
    assert op == "evaluate", op
    r, c = case["rows"], case["cols"]
    return dict(x=_randn(g, (r, c), case["x"], 2.0), t=_targets(g, (r,), c, 0.0))


def _to_supa(src):
    src = src.contiguous()
    dst = torch.empty(src.shape, dtype=src.dtype, device="supa")
    if src.numel():
        torch_supa._C.memcpy_d2d(dst.data_ptr(), src.data_ptr(), src.numel() * src.element_size())
    return dst


STEP, LR, BETAS, EPS, WD, CLIP = 10.0, 1e-4, (0.9, 0.999), 1e-8, 0.01, 1.0
GRAD_OF = {"bias_act": ("x", "bias"), "gated": ("x",), "cross_entropy": ("x",), "pixel_loss": ("x",),
           "attention": ("x",), "norm": ("x", "w", "b"), "pointwise_loss": ("x",)}


def prepare(case, seed):
    src = _inputs(case, seed)
    torch.cuda.synchronize()
    d = {k: _to_supa(v) for k, v in src.items()}
    torch.supa.synchronize()
    del src
    if case["op"] == "optimizer":
        n = len(_optimizer_shapes(case))
        params = [d["p%d" % i].requires_grad_() for i in range(n)]
        opt = torch.optim.AdamW(params, lr=LR, betas=BETAS, eps=EPS, weight_decay=WD,
                                **({"fused": True} if case["fused"] else {"foreach": True}))
        for i, p in enumerate(params):
            p.grad = d["g%d" % i]
            step = torch.tensor(STEP, device="supa" if case["fused"] else "cpu")
            opt.state[p] = {"step": step, "exp_avg": d["m%d" % i], "exp_avg_sq": d["v%d" % i]}
        return {"case": case, "params": params, "opt": opt}
    if case["op"] == "bias_act" and case["layout"] == "transposed":
        d["x"] = d["x"].t()
        if "gy" in d:
            d["gy"] = d["gy"].t()
    if case.get("train", True):
        for k in GRAD_OF.get(case["op"], ()):
            d[k] = d[k].requires_grad_()
    d["case"] = case
    return d


# --------------------------------------------------------------- formulas
def _forward(case, d):
    """The case's forward, as a program writes it: the output that the
    gradient starts from."""
    op = case["op"]
    if op == "bias_act":
        return ACTS[case["act"]](d["x"] + d["bias"])
    if op == "gated":
        gate, up = d["x"].chunk(2, dim=-1)
        return F.silu(gate) * up
    if op == "cross_entropy":
        return F.cross_entropy(d["x"], d["t"], ignore_index=IGNORE, reduction=case["reduction"])
    if op == "pixel_loss":
        return F.cross_entropy(d["x"], d["t"], weight=d.get("weight"), ignore_index=IGNORE)
    if op == "attention":
        return F.softmax(d["x"].masked_fill(d["mask"], -math.inf), dim=-1)
    if op == "norm":
        x = d["x"]
        var, mean = torch.var_mean(x, dim=-1 if case["inner"] == 1 else (0, 2), correction=0, keepdim=True)
        return (x - mean) * torch.rsqrt(var + 1e-5) * d["w"] + d["b"]
    assert op == "pointwise_loss", op
    kind, red = case["kind"], case["reduction"]
    if kind == "bce":
        return F.binary_cross_entropy_with_logits(d["x"], d["t"], pos_weight=d["pw"], reduction=red)
    return {"mse": F.mse_loss, "smooth_l1": F.smooth_l1_loss, "huber": F.huber_loss}[kind](d["x"], d["t"],
                                                                                      reduction=red)


def _evaluate(x, t, dtype):
    top, pred = x.max(dim=-1)
    return top, pred, (pred == t).to(dtype).mean(), x.mean(dim=0)


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "optimizer":
        params, opt = state["params"], state["opt"]
        norm = torch.nn.utils.clip_grad_norm_(params, CLIP)
        opt.step()
        s = [opt.state[p] for p in params]
        return norm, [p.detach() for p in params], [v["exp_avg"] for v in s], [v["exp_avg_sq"] for v in s]
    if op == "evaluate":
        return _evaluate(state["x"], state["t"], torch.float32)
    if not case.get("train", True):
        with torch.no_grad():
            return _forward(case, state)
    leaves = [state[k] for k in GRAD_OF[op]]
    for p in leaves:
        p.grad = None
    y = _forward(case, state)
    y.backward(state.get("gy"))
    return y.detach(), [p.grad for p in leaves]


def exact(case, seed):
    op = case["op"]
    src = _inputs(case, seed)
    if op == "optimizer":
        n = len(_optimizer_shapes(case))
        p, g, m, v = ([src["%s%d" % (k, i)].double() for i in range(n)] for k in "pgmv")
        norm = torch.sqrt(sum(t.square().sum() for t in g))
        coef = torch.clamp(CLIP / (norm + 1e-6), max=1.0)
        bc1, bc2 = 1 - BETAS[0] ** (STEP + 1), 1 - BETAS[1] ** (STEP + 1)
        for i in range(n):
            gi = g[i] * coef
            p[i] = p[i] * (1 - LR * WD)
            m[i] = m[i] * BETAS[0] + gi * (1 - BETAS[0])
            v[i] = v[i] * BETAS[1] + gi * gi * (1 - BETAS[1])
            p[i] = p[i] - LR / bc1 * m[i] / (v[i].sqrt() / math.sqrt(bc2) + EPS)
        return norm, p, m, v
    d = {k: v.double() if v.is_floating_point() else v for k, v in src.items()}
    del src
    if op == "evaluate":
        top, pred, acc, mean = _evaluate(d["x"], d["t"], torch.float64)
        return top, None, acc, mean
    if op == "bias_act" and case["layout"] == "transposed":
        d["x"] = d["x"].t()
        if "gy" in d:
            d["gy"] = d["gy"].t()
    y = _forward(case, d)
    if not case.get("train", True):
        return y
    return y, _gradients(case, d, y)


def _gradients(case, d, y):
    """The gradients of GRAD_OF[op], by their formulas (torch's autograd
    cannot run on its HIP device in a process where supa is the accelerator)."""
    op, x, gy = case["op"], d["x"], d.get("gy")
    if op == "bias_act":
        u = x + d["bias"]
        if case["act"] == "relu":
            gx = gy * (u > 0)
        elif case["act"] == "silu":
            gx = torch.ops.aten.silu_backward(gy, u)
        else:
            gx = torch.ops.aten.gelu_backward(gy, u, approximate="tanh" if case["act"] == "gelu_tanh" else "none")
        return [gx, gx.sum(0)]
    if op == "gated":
        gate, up = x.chunk(2, dim=-1)
        return [torch.cat([torch.ops.aten.silu_backward(gy * up, gate), gy * F.silu(gate)], dim=-1)]
    if op in ("cross_entropy", "pixel_loss"):
        t = d["t"]
        kept = t != IGNORE
        w = kept.double() if d.get("weight") is None else d["weight"][t.clamp(min=0)] * kept
        if case.get("reduction", "mean") == "mean":
            scale = w / w.sum()
        else:
            scale = w * gy if gy is not None else w
        gx = F.softmax(x, dim=1) * scale.unsqueeze(1)
        gx.scatter_add_(1, t.clamp(min=0).unsqueeze(1), -scale.unsqueeze(1))
        return [gx]
    if op == "attention":
        return [y * (gy - (gy * y).sum(-1, keepdim=True))]
    if op == "norm":
        dims = -1 if case["inner"] == 1 else (0, 2)
        var, mean = torch.var_mean(x, dim=dims, correction=0, keepdim=True)
        rstd = torch.rsqrt(var + 1e-5)
        xh = (x - mean) * rstd
        gh = gy * d["w"]
        gx = rstd * (gh - gh.mean(dims, keepdim=True) - xh * (gh * xh).mean(dims, keepdim=True))
        return [gx, (gy * xh).sum_to_size(d["w"].shape), gy.sum_to_size(d["b"].shape)]
    assert op == "pointwise_loss", op
    t, e = d["t"], x - d["t"]
    if case["kind"] == "mse":
        gx = 2 * e
    elif case["kind"] == "bce":
        s = torch.sigmoid(x)
        gx = s * (1 + (d["pw"] - 1) * t) - d["pw"] * t
    else:
        gx = e.clamp(-1, 1)  # smooth_l1 and huber agree at beta = delta = 1
    if case["reduction"] == "mean":
        gx = gx / gx.numel()
    return [gx if gy is None else gx * gy]


# ------------------------------------------------------------ bookkeeping
def work(case):
    """Bytes that one pass cannot do without: each input read once and each
    output written once, for the forward and for the backward."""
    op = case["op"]
    if op == "optimizer":
        n = sum(math.prod(s) for s in _optimizer_shapes(case))
        return {"bytes": (4 + 28) * n, "flops": 20 * n}  # the norm's read, then p, g, m, v in and p, m, v out
    e = SIZE[case["x"]]
    if op == "bias_act":
        n, c = case["rows"] * case["cols"], case["cols"]
        o, eb = max(e, SIZE[case["bias"]]), SIZE[case["bias"]]
        nbytes = n * (e + o) + c * eb
        if case["train"]:
            nbytes += n * (e + o + e) + 2 * c * eb  # x and gy in, gx out, bias in, its gradient out
        return {"bytes": nbytes, "flops": 20 * n}
    if op == "gated":
        n = case["rows"] * case["cols"]
        return {"bytes": e * (3 * n + 5 * n), "flops": 20 * n}
    if op == "cross_entropy":
        n = case["rows"] * case["cols"]
        return {"bytes": 3 * e * n + 16 * case["rows"], "flops": 10 * n}
    if op == "pixel_loss":
        s = case["batch"] * case["height"] * case["width"]
        return {"bytes": 3 * e * s * case["cols"] + 16 * s, "flops": 10 * s * case["cols"]}
    if op == "attention":
        n = case["batch"] * case["heads"] * case["rows"] * case["cols"]
        return {"bytes": e * (2 * n + 3 * n) + 2 * case["rows"] * case["cols"], "flops": 10 * n}
    if op == "norm":
        n = case["rows"] * case["cols"] * case["inner"]
        return {"bytes": e * (2 * n + 3 * n) + 6 * e * case["cols"], "flops": 20 * n}
    if op == "pointwise_loss":
        n = case["rows"] * case["cols"]
        none = case["reduction"] == "none"
        nbytes = e * ((3 if none else 2) * n + (4 if none else 3) * n)
        return {"bytes": nbytes + (2 * e * case["cols"] if case["kind"] == "bce" else 0), "flops": 15 * n}
    n = case["rows"] * case["cols"]
    return {"bytes": e * n + (e + 16) * case["rows"] + e * case["cols"], "flops": 2 * n}


def tolerance(case):
    op = case["op"]
    if op == "optimizer":
        return {"rel": 1e-5, "max": 1e-3}
    if op == "evaluate":
        return {"rel": 1e-5 if case["x"] == "f32" else 4e-3, "differ": 0.0}
    return {"rel": 1e-5, "max": 1e-3} if case["x"] == "f32" else {"rel": 1e-2, "max": 0.2}
