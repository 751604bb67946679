"""The work that the framework's users have it do, as timed cases.

Each case goes through the public entry points (the C ABI through
``lanternl_amd._lib.call``, ``lanternl_amd.kernels`` and
``lanternl_amd.lmtrain``).  Seven kinds of pass:

  linear     a linear layer over `tokens` rows: Y = X.W, dX = dY.W^T and
             dW = X^T.dY (the three products of a forward and backward)
  decode     one product of a few rows with a large weight (token generation)
  head       logits = H.W, the fused softmax + cross-entropy with dlogits
             written over the logits, dW = H^T.dlogits, dH = dlogits.W^T
  attention  causal attention composed of the batched products and the row
             softmax, forward and backward, q/k/v as [batch*heads][seq][head_dim]
  rows       RMSNorm, RoPE, SwiGLU and row softmax, forward and backward
  embed      embedding lookup, its scatter-add backward and an AdamW step on
             the table, token ids with the skew of natural text
  lm         LMTrain's batch loop: a batch handed over and one optimizer step,
             `steps` times, then the last losses and the updated parameters
  host       the flat-table products on host doubles, as a Lua host calls them
"""
import ctypes
import math

import numpy as np
import torch

from lanternl_amd import device, kernels, lmtrain
from lanternl_amd._lib import call

EPS = 1e-6
ADAM = dict(lr=1e-4, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.01, clip_norm=1.0, step=10)


def listed():
    return [
        # the smallest layer in use: 256 tokens, dim 128 -> ffn 256 (three launches' latency)
        {"name": "linear_256x128x256", "kind": "linear", "tokens": 256, "din": 128, "dout": 256},
        # an ordinary layer whose sizes fit no tile: a ragged token count, dim 768, an odd width
        {"name": "linear_1999x768x2050", "kind": "linear", "tokens": 1999, "din": 768, "dout": 2050},
        # the large square products
        {"name": "linear_4096", "kind": "linear", "tokens": 4096, "din": 4096, "dout": 4096},
        # a token each for sixteen sequences being generated
        {"name": "decode_16x4096x4096", "kind": "decode", "rows": 16, "k": 4096, "n": 4096},
        # the language-model head over a full-size vocabulary
        {"name": "head_512x128x32000", "kind": "head", "tokens": 512, "dim": 128, "vocab": 32000},
        # eight windows of 256 tokens, eight heads of 64
        {"name": "attention_64x256x64", "kind": "attention", "batch": 64, "seq": 256, "head_dim": 64},
        # the bandwidth-bound layers at 4096 tokens
        {"name": "rows_4096x1024x4096", "kind": "rows", "tokens": 4096, "heads": 16, "head_dim": 64, "ffn": 4096},
        # the table of a 32000-word vocabulary: lookup, gradient and update
        {"name": "embed_32000x256", "kind": "embed", "vocab": 32000, "dim": 256, "tokens": 2048},
        # a character model on short windows: the smallest training loop
        {"name": "lm_tiny", "kind": "lm", "vocab": 256, "dim": 64, "layers": 2, "heads": 4, "ffn": 128,
         "batch": 4, "seq": 32, "opt": "sgd", "ragged": True, "steps": 32},
        # the benchmark's training loop
        {"name": "lm_2000x128x4", "kind": "lm", "vocab": 2000, "dim": 128, "layers": 4, "heads": 8, "ffn": 256,
         "batch": 8, "seq": 64, "opt": "sgd", "ragged": False, "steps": 32},
        # a larger model on longer windows, the trainer's default optimizer, the last window short
        {"name": "lm_4000x512x4", "kind": "lm", "vocab": 4000, "dim": 512, "layers": 4, "heads": 8, "ffn": 1024,
         "batch": 8, "seq": 256, "opt": "adamw", "ragged": True, "steps": 16},
        # the three products of the smallest layer on a Lua host's double tables
        {"name": "host_256x128x256", "kind": "host", "tokens": 256, "din": 128, "dout": 256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "decode", "head", "attention", "rows", "embed", "lm", "lm", "host"])
    if kind == "linear":
        return {"kind": kind, "tokens": _log(rng, 64, 4096), "din": _log(rng, 64, 4096), "dout": _log(rng, 64, 4096)}
    if kind == "decode":
        return {"kind": kind, "rows": _log(rng, 1, 64), "k": _log(rng, 512, 4096), "n": _log(rng, 512, 4096)}
    if kind == "head":
        return {"kind": kind, "tokens": _log(rng, 64, 1024), "dim": _log(rng, 64, 512), "vocab": _log(rng, 1000, 32000)}
    if kind == "attention":
        return {"kind": kind, "batch": _log(rng, 8, 128), "seq": _log(rng, 32, 512), "head_dim": rng.choice([16, 32, 64, 128])}
    if kind == "rows":
        return {"kind": kind, "tokens": _log(rng, 64, 4096), "heads": rng.randint(1, 16),
                "head_dim": rng.choice([16, 32, 64, 128]), "ffn": _log(rng, 128, 4096)}
    if kind == "embed":
        return {"kind": kind, "vocab": _log(rng, 256, 32000), "dim": _log(rng, 64, 512), "tokens": _log(rng, 64, 4096)}
    if kind == "lm":
        heads, hd = rng.randint(1, 8), rng.choice([16, 32, 64])
        return {"kind": kind, "vocab": _log(rng, 64, 4000), "dim": heads * hd, "layers": rng.randint(1, 4), "heads": heads,
                "ffn": heads * hd * 2 + 4 * rng.randint(0, 15), "batch": _log(rng, 1, 8), "seq": _log(rng, 16, 256),
                "opt": rng.choice(["sgd", "adamw"]), "ragged": rng.random() < 0.5, "steps": 16}
    return {"kind": kind, "tokens": _log(rng, 32, 1024), "din": _log(rng, 32, 1024), "dout": _log(rng, 32, 1024)}


# ---- inputs -----------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).add_(mean)


def _empty(*shape):
    return torch.empty(*shape, device="cuda", dtype=torch.float32)


def _linear_inputs(c, seed):
    g = _gen(seed)
    return (_randn(g, c["tokens"], c["din"]), _randn(g, c["din"], c["dout"], std=0.02),
            _randn(g, c["tokens"], c["dout"], std=1e-3))


def _decode_inputs(c, seed):
    g = _gen(seed)
    return _randn(g, c["rows"], c["k"]), _randn(g, c["k"], c["n"], std=0.02)


def _head_inputs(c, seed):
    g = _gen(seed)
    h, w = _randn(g, c["tokens"], c["dim"]), _randn(g, c["dim"], c["vocab"], std=0.02)
    return h, w, torch.randint(c["vocab"], (c["tokens"],), generator=g, device="cuda", dtype=torch.int32)


def _attention_inputs(c, seed):
    g = _gen(seed)
    shape = (c["batch"], c["seq"], c["head_dim"])
    return [_randn(g, *shape) for _ in range(4)]   # q, k, v, dctx


def _rows_inputs(c, seed):
    g = _gen(seed)
    n, d, f = c["tokens"], c["heads"] * c["head_dim"], c["ffn"]
    return {"x": _randn(g, n, d), "w": _randn(g, d, std=0.1, mean=1.0), "dy": _randn(g, n, d),
            "q": _randn(g, n, d), "dq": _randn(g, n, d),
            "gate": _randn(g, n, f), "up": _randn(g, n, f), "dout": _randn(g, n, f),
            "s": _randn(g, n, f, std=2.0), "dp": _randn(g, n, f)}


def _embed_inputs(c, seed):
    g = _gen(seed)
    v, d, n = c["vocab"], c["dim"], c["tokens"]
    # log-uniform ranks: a few words make up most of a text
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    ids = (torch.exp(u * math.log(v)) - 1.0).floor().clamp_(0, v - 1).to(torch.int32)
    return {"table": _randn(g, v, d, std=0.02), "ids": ids, "dout": _randn(g, n, d, std=1e-3),
            "m": _randn(g, v, d, std=1e-4), "v": _randn(g, v, d, std=1e-4).square_().add_(1e-10)}


def _lm_inputs(c, seed):
    rng = np.random.default_rng(int(seed))
    cfg = lmtrain.config(c["vocab"], c["dim"], c["layers"], c["heads"], c["ffn"], c["batch"], c["seq"])
    params = lmtrain.init_params(cfg, rng)
    batches = []
    for _ in range(c["steps"]):
        ids = rng.integers(0, c["vocab"], (c["batch"], c["seq"] + 1), dtype=np.int32)
        lens = np.full(c["batch"], c["seq"], np.int32)
        if c["ragged"]:
            lens[-1] = rng.integers(max(1, c["seq"] // 4), c["seq"] + 1)
        batches.append((np.ascontiguousarray(ids[:, :-1]), np.ascontiguousarray(ids[:, 1:]), lens))
    return cfg, params, batches


def _host_inputs(c, seed):
    rng = np.random.default_rng(int(seed))
    return (rng.uniform(-1, 1, (c["tokens"], c["din"])), rng.uniform(-1, 1, (c["din"], c["dout"])),
            rng.uniform(-1, 1, (c["tokens"], c["dout"])))


def prepare(case, seed):
    device.init(0)
    s = {"case": case}
    kind = case["kind"]
    if kind == "linear":
        x, w, dy = _linear_inputs(case, seed)
        s.update(x=x, w=w, dy=dy, y=torch.empty_like(dy), dx=torch.empty_like(x), dw=torch.empty_like(w))
    elif kind == "decode":
        x, w = _decode_inputs(case, seed)
        s.update(x=x, w=w, y=_empty(case["rows"], case["n"]))
    elif kind == "head":
        h, w, t = _head_inputs(case, seed)
        s.update(h=h, w=w, t=t, logits=_empty(case["tokens"], case["vocab"]), losses=_empty(case["tokens"]),
                 dw=torch.empty_like(w), dh=torch.empty_like(h))
    elif kind == "attention":
        q, k, v, do = _attention_inputs(case, seed)
        b, t = case["batch"], case["seq"]
        s.update(q=q, k=k, v=v, do=do, s=_empty(b, t, t), p=_empty(b, t, t), dp=_empty(b, t, t), ds=_empty(b, t, t),
                 ctx=torch.empty_like(q), dq=torch.empty_like(q), dk=torch.empty_like(q), dv=torch.empty_like(q))
    elif kind == "rows":
        s.update(_rows_inputs(case, seed))
        n, d = s["x"].shape
        s.update(y=_empty(n, d), inv=_empty(n), dx=_empty(n, d), dw=_empty(d))
        for name in ("act", "dgate", "dup", "p", "ds"):
            s[name] = torch.empty_like(s["gate"])
    elif kind == "embed":
        s.update(_embed_inputs(case, seed))
        s.update(out=torch.empty_like(s["dout"]), grad=torch.empty_like(s["table"]),
                 ss=torch.empty(1, device="cuda", dtype=torch.float64))
    elif kind == "lm":
        cfg, params, batches = _lm_inputs(case, seed)
        step = lmtrain.GpuLMStep(case["vocab"], case["dim"], case["layers"], case["heads"], case["ffn"], case["batch"],
                                 case["seq"])
        step.set_params(params)
        s.update(step=step, batches=batches)
    else:
        x, w, dy = _host_inputs(case, seed)
        s.update(x=x, w=w, dy=dy, y=np.zeros_like(dy), dx=np.zeros_like(x), dw=np.zeros_like(w))
    torch.cuda.synchronize()   # the inputs are made on torch's stream, the library has its own
    return s


# ---- the passes -------------------------------------------------------------
def run(s):
    return globals()["_run_" + s["case"]["kind"]](s, s["case"])


def _run_linear(s, c):
    n, i, o = c["tokens"], c["din"], c["dout"]
    x, w, dy, y, dx, dw = (s[k].data_ptr() for k in ("x", "w", "dy", "y", "dx", "dw"))
    kernels.sgemm_raw(0, 0, n, o, i, 1.0, x, i, w, o, 0.0, y, o)
    kernels.sgemm_raw(0, 1, n, i, o, 1.0, dy, o, w, o, 0.0, dx, i)
    kernels.sgemm_raw(1, 0, i, o, n, 1.0, x, i, dy, o, 0.0, dw, o)
    return {"y": s["y"], "dx": s["dx"], "dw": s["dw"]}


def _run_decode(s, c):
    kernels.sgemm_raw(0, 0, c["rows"], c["n"], c["k"], 1.0, s["x"].data_ptr(), c["k"], s["w"].data_ptr(), c["n"], 0.0,
                      s["y"].data_ptr(), c["n"])
    return s["y"]


def _run_head(s, c):
    n, d, v = c["tokens"], c["dim"], c["vocab"]
    h, w, t, lg, ls, dw, dh = (s[k].data_ptr() for k in ("h", "w", "t", "logits", "losses", "dw", "dh"))
    kernels.sgemm_raw(0, 0, n, v, d, 1.0, h, d, w, v, 0.0, lg, v)
    call("lhip_ce_fused", lg, t, ls, lg, n, v, -1, 1.0 / n)
    kernels.sgemm_raw(1, 0, d, v, n, 1.0, h, d, lg, v, 0.0, dw, v)
    kernels.sgemm_raw(0, 1, n, d, v, 1.0, lg, v, w, v, 0.0, dh, d)
    return {"losses": s["losses"], "dlogits": s["logits"], "dw": s["dw"], "dh": s["dh"]}


def _run_attention(s, c):
    b, t, d = c["batch"], c["seq"], c["head_dim"]
    td, tt, scale = t * d, t * t, 1.0 / math.sqrt(d)
    q, k, v, do, sc, p, dp, ds, ctx, dq, dk, dv = (
        s[x].data_ptr() for x in ("q", "k", "v", "do", "s", "p", "dp", "ds", "ctx", "dq", "dk", "dv"))
    mm = kernels.sgemm_strided_batched
    mm(0, 1, t, t, d, 1.0, q, d, td, k, d, td, 0.0, sc, t, tt, b)
    call("lhip_softmax_fwd", sc, p, b * t, t, scale, 1, 0, t)
    mm(0, 0, t, d, t, 1.0, p, t, tt, v, d, td, 0.0, ctx, d, td, b)
    mm(0, 1, t, t, d, 1.0, do, d, td, v, d, td, 0.0, dp, t, tt, b)
    mm(1, 0, t, d, t, 1.0, p, t, tt, do, d, td, 0.0, dv, d, td, b)
    call("lhip_softmax_bwd", p, dp, ds, b * t, t, scale, 1, 0, t, 0)
    mm(0, 0, t, d, t, 1.0, ds, t, tt, k, d, td, 0.0, dq, d, td, b)
    mm(1, 0, t, d, t, 1.0, ds, t, tt, q, d, td, 0.0, dk, d, td, b)
    return {"p": s["p"], "ctx": s["ctx"], "dq": s["dq"], "dk": s["dk"], "dv": s["dv"]}


def _run_rows(s, c):
    n, d, f, h, hd = c["tokens"], c["heads"] * c["head_dim"], c["ffn"], c["heads"], c["head_dim"]
    a = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
    call("lhip_rmsnorm_fwd", a["x"], a["w"], a["y"], a["inv"], n, d, EPS)
    call("lhip_rope", a["q"], None, n, h, hd, d, 0, 0, 10000.0, 1, 0)
    call("lhip_swiglu_fwd", a["gate"], f, a["up"], f, a["act"], f, n, f)
    call("lhip_softmax_fwd", a["s"], a["p"], n, f, 1.0, 0, 0, 0)
    call("lhip_softmax_bwd", a["p"], a["dp"], a["ds"], n, f, 1.0, 0, 0, 0, 0)
    call("lhip_swiglu_bwd", a["gate"], f, a["up"], f, a["dout"], f, a["dgate"], f, a["dup"], f, n, f, 0)
    call("lhip_rope", a["dq"], None, n, h, hd, d, 0, 0, 10000.0, 1, 1)
    call("lhip_rmsnorm_bwd", a["x"], a["w"], a["inv"], a["dy"], a["dx"], a["dw"], n, d, 0)
    return {k: s[k] for k in ("y", "inv", "q", "act", "p", "ds", "dgate", "dup", "dq", "dx", "dw")}


def _run_embed(s, c):
    v, d, n = c["vocab"], c["dim"], c["tokens"]
    t, i, do, out, g, m, vv, ss = (s[k].data_ptr() for k in ("table", "ids", "dout", "out", "grad", "m", "v", "ss"))
    call("lhip_embed_fwd", t, i, out, n, d, v)
    call("lhip_embed_bwd", do, i, g, n, d, v, 1.0, 0)
    call("lhip_sumsq", g, v * d, ss)
    call("lhip_adamw_step", t, g, m, vv, v * d, ss, ADAM["lr"], ADAM["beta1"], ADAM["beta2"], ADAM["eps"],
         ADAM["weight_decay"], 1.0, ADAM["clip_norm"], ADAM["step"], None, None)
    return {k: s[k] for k in ("out", "grad", "table", "m", "v")}


def _run_lm(s, c):
    step = s["step"]
    for ids, tgt, lens in s["batches"]:
        step.set_batch(ids, tgt, lens if c["ragged"] else None)
        if c["opt"] == "sgd":
            step.step(1e-2, 0.9, 0.01, 1.0)
        else:
            step.step_adamw(1e-4)
    return {"losses": step.stats()["window_losses"], "params": step.params()}


def _run_host(s, c):
    n, i, o = c["tokens"], c["din"], c["dout"]
    x, w, dy, y, dx, dw = (s[k].ctypes.data_as(ctypes.c_void_p) for k in ("x", "w", "dy", "y", "dx", "dw"))
    call("lhip_matmul_host", 0, x, w, y, n, i, o, 0)
    call("lhip_matmul_host", 1, dy, w, dx, n, o, i, 0)
    call("lhip_matmul_host", 2, x, dy, dw, n, i, o, 0)
    return {"y": s["y"], "dx": s["dx"], "dw": s["dw"]}


# ---- what a pass cannot do without -------------------------------------------
def work(case):
    c, kind = case, case["kind"]
    if kind in ("linear", "host"):
        n, i, o = c["tokens"], c["din"], c["dout"]
        size = 4 if kind == "linear" else 8
        return {"bytes": size * 2 * (n * i + i * o + n * o), "flops": 6 * n * i * o}
    if kind == "decode":
        m, k, n = c["rows"], c["k"], c["n"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    if kind == "head":
        n, d, v = c["tokens"], c["dim"], c["vocab"]
        return {"bytes": 4 * (2 * n * d + 2 * d * v + n * v + 2 * n), "flops": 6 * n * d * v}
    if kind == "attention":
        b, t, d = c["batch"], c["seq"], c["head_dim"]
        half = b * t * (t + 1) // 2   # the causal scores
        return {"bytes": 4 * (8 * b * t * d + b * t * t), "flops": 12 * half * d}
    if kind == "rows":
        n, d, f = c["tokens"], c["heads"] * c["head_dim"], c["ffn"]
        # per element: RMSNorm 2 + 3 (x is read by both), RoPE 2 x 2, SwiGLU 3 + 5, softmax 2 + 3
        return {"bytes": 4 * (9 * n * d + 13 * n * f + 2 * n + 3 * d), "flops": n * (20 * d + 30 * f)}
    if kind == "embed":
        v, d, n = c["vocab"], c["dim"], c["tokens"]
        return {"bytes": 4 * (7 * v * d + 3 * n * d + 2 * n), "flops": 15 * v * d}
    n, d, f, v, t = c["batch"] * c["seq"], c["dim"], c["ffn"], c["vocab"], c["seq"]
    mats = c["layers"] * (4 * d * d + 3 * d * f) + v * d
    attn = c["layers"] * 12 * n * (t + 1) // 2 * d
    state = 2 if c["opt"] == "sgd" else 3
    acts = c["layers"] * n * (6 * d + 3 * f) + n * v
    return {"bytes": c["steps"] * 4 * (mats * 2 * state + 2 * acts) + 4 * mats,
            "flops": c["steps"] * (6 * n * mats + attn)}


def tolerance(case):
    # 32-bit sums: four times what the products and row kernels are off 64 bits,
    # and for `lm` what a whole run of optimizer steps is.  AdamW's first steps
    # move a weight by lr * sign(gradient), so the few weights whose gradient is
    # near zero move the other way after any change of rounding: a few steps of
    # 1e-4 on weights of 0.02
    if case["kind"] == "lm" and case["opt"] == "adamw":
        return {"rel": 5e-6, "max": 0.05}
    return {"linear": {"rel": 4e-6}, "decode": {"rel": 2e-6}, "head": {"rel": 4e-6}, "attention": {"rel": 4e-6},
            "rows": {"rel": 4e-6}, "embed": {"rel": 4e-6}, "lm": {"rel": 5e-6}, "host": {"rel": 2e-6}}[case["kind"]]


# ---- the same results in 64 bits -----------------------------------------------
def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


def _exact_linear(c, seed):
    x, w, dy = (a.double() for a in _linear_inputs(c, seed))
    return {"y": x @ w, "dx": dy @ w.t(), "dw": x.t() @ dy}


def _exact_decode(c, seed):
    x, w = _decode_inputs(c, seed)
    return x.double() @ w.double()


def _exact_head(c, seed):
    h, w, t = _head_inputs(c, seed)
    h, w, t = h.double(), w.double(), t.long()
    n = c["tokens"]
    z = h @ w
    lse = torch.logsumexp(z, 1)
    losses = lse - z.gather(1, t[:, None])[:, 0]
    dz = torch.exp(z - lse[:, None])
    dz[torch.arange(n, device=dz.device), t] -= 1.0
    dz /= n
    return {"losses": losses, "dlogits": dz, "dw": h.t() @ dz, "dh": dz @ w.t()}


def _exact_attention(c, seed):
    q, k, v, do = (a.double() for a in _attention_inputs(c, seed))
    t, scale = c["seq"], 1.0 / math.sqrt(c["head_dim"])
    keep = torch.ones(t, t, dtype=torch.bool, device="cuda").tril()
    tr = lambda a: a.transpose(1, 2).contiguous()   # noqa: E731
    p = torch.softmax((q @ tr(k) * scale).masked_fill(~keep, -math.inf), -1)
    dp = do @ tr(v)
    ds = scale * p * (dp - (dp * p).sum(-1, keepdim=True))
    return {"p": p, "ctx": p @ v, "dq": ds @ k, "dk": tr(ds) @ q, "dv": tr(p) @ do}


def _rotate(x, heads, hd, sign):
    n = x.shape[0]
    inv = 10000.0 ** (-2.0 * torch.arange(hd // 2, device=x.device, dtype=torch.float64) / hd)
    ang = torch.arange(n, device=x.device, dtype=torch.float64)[:, None] * inv
    cs, sn = torch.cos(ang)[:, None], sign * torch.sin(ang)[:, None]
    y = x.view(n, heads, hd // 2, 2)
    return torch.stack((y[..., 0] * cs - y[..., 1] * sn, y[..., 0] * sn + y[..., 1] * cs), -1).reshape(n, heads * hd)


def _exact_rows(c, seed):
    a = {k: v.double() for k, v in _rows_inputs(c, seed).items()}
    inv = 1.0 / torch.sqrt(a["x"].square().mean(1) + EPS)
    xn, g = a["x"] * inv[:, None], a["dy"] * a["w"]
    dx = inv[:, None] * (g - xn * (g * xn).mean(1, keepdim=True))
    sg = torch.sigmoid(a["gate"])
    p = torch.softmax(a["s"], 1)
    return {"y": xn * a["w"], "inv": inv, "q": _rotate(a["q"], c["heads"], c["head_dim"], 1.0),
            "act": a["gate"] * sg * a["up"], "p": p, "ds": p * (a["dp"] - (a["dp"] * p).sum(1, keepdim=True)),
            "dgate": sg * (1 + a["gate"] * (1 - sg)) * a["up"] * a["dout"], "dup": a["gate"] * sg * a["dout"],
            "dq": _rotate(a["dq"], c["heads"], c["head_dim"], -1.0), "dx": dx, "dw": (a["dy"] * xn).sum(0)}


def _exact_embed(c, seed):
    a = _embed_inputs(c, seed)
    ids, a = a["ids"].long(), {k: v.double() for k, v in a.items() if k != "ids"}
    g = torch.zeros_like(a["table"]).index_add_(0, ids, a["dout"])
    norm = g.norm()
    if norm > ADAM["clip_norm"]:
        g = g * (ADAM["clip_norm"] / norm)
    b1, b2 = ADAM["beta1"], ADAM["beta2"]
    m, v = b1 * a["m"] + (1 - b1) * g, b2 * a["v"] + (1 - b2) * g * g
    t = a["table"] * (1 - ADAM["lr"] * ADAM["weight_decay"])
    t = t - ADAM["lr"] / (1 - b1 ** ADAM["step"]) * m / (torch.sqrt(v / (1 - b2 ** ADAM["step"])) + ADAM["eps"])
    return {"out": a["table"][ids], "grad": g, "table": t, "m": m, "v": v}


def _lm_losses(c, cfg, table, flat, ids, tgt, lens):
    """Each window's mean cross-entropy, from the flat parameters, in 64 bits."""
    P = {name: flat[off:off + r * k].view(r, k) for name, off, r, k in table}
    b, t, h, d = c["batch"], c["seq"], c["heads"], c["dim"]
    hd = d // h
    inv = cfg.rope_base ** (-2.0 * torch.arange(hd // 2, device="cuda", dtype=torch.float64) / hd)
    ang = torch.arange(t, device="cuda", dtype=torch.float64)[:, None] * inv
    cs, sn = torch.cos(ang)[None, :, None], torch.sin(ang)[None, :, None]
    keep = torch.ones(t, t, dtype=torch.bool, device="cuda").tril()

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + cfg.eps) * w

    def split(x, rope):
        x = x.view(b, t, h, hd)
        if rope:
            y = x.view(b, t, h, hd // 2, 2)
            x = torch.stack((y[..., 0] * cs - y[..., 1] * sn, y[..., 0] * sn + y[..., 1] * cs), -1).reshape(b, t, h, hd)
        return x.permute(0, 2, 1, 3).reshape(b * h, t, hd)

    x = P["emb"][ids]
    for l in range(c["layers"]):
        y = norm(x, P[f"ln1.{l}"])
        q, k, v = (split(y @ P[f"{w}.{l}"], w != "wv") for w in ("wq", "wk", "wv"))
        sc = (q @ k.transpose(1, 2).contiguous() / math.sqrt(hd)).masked_fill(~keep, -math.inf)
        o = (torch.softmax(sc, -1) @ v).view(b, h, t, hd).permute(0, 2, 1, 3).reshape(b * t, d)
        x = x + o @ P[f"wo.{l}"]
        y = norm(x, P[f"ln2.{l}"])
        x = x + (torch.nn.functional.silu(y @ P[f"w1.{l}"]) * (y @ P[f"w3.{l}"])) @ P[f"w2.{l}"]
    z = norm(x, P["lnf"]) @ P["emb"].t()
    ce = torch.nn.functional.cross_entropy(z, tgt, reduction="none").view(b, t)
    used = torch.arange(t, device="cuda")[None] < lens[:, None]
    return (ce * used).sum(1) / lens


def _exact_lm(c, seed):
    cfg, params, batches = _lm_inputs(c, seed)
    table = lmtrain.param_table(cfg)
    p = torch.from_numpy(params).cuda().double()
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    for step, (ids, tgt, lens) in enumerate(batches, 1):
        ids, tgt = (torch.from_numpy(a).cuda().long().reshape(-1) for a in (ids, tgt))
        flat = p.clone().requires_grad_(True)
        losses = _lm_losses(c, cfg, table, flat, ids, tgt, torch.from_numpy(lens).cuda())
        g, = torch.autograd.grad(losses.mean(), flat)
        norm = g.norm()
        if norm > 1.0:
            g = g / norm
        if c["opt"] == "sgd":
            g = g + 0.01 * p
            m = 0.9 * m + g
            p = p - 1e-2 * m
        else:
            m, v = 0.9 * m + 0.1 * g, 0.95 * v + 0.05 * g * g
            p = p * (1 - 1e-4 * 0.01)
            p = p - 1e-4 / (1 - 0.9 ** step) * m / (torch.sqrt(v / (1 - 0.95 ** step)) + 1e-8)
    return {"losses": losses.detach(), "params": p}


def _exact_host(c, seed):
    x, w, dy = (torch.from_numpy(a).cuda() for a in _host_inputs(c, seed))
    return {"y": x @ w, "dx": dy @ w.t(), "dw": x.t() @ dy}
