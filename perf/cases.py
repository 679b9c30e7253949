"""What a user of this framework has it do, as timed cases through its public
entry points: matrix products, the layers around them (linear, norms, softmax,
reductions, attention) forward and backward, a multi-head attention layer and
a transformer block on a lazy HIP stream, and the decoder's generate.

Device operands live in torch tensors, whose addresses the direct entry points
take; work goes to the null stream, torch's own. The lazy stream's results and
the decoder's come back as numpy arrays, the only form those entry points give.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from oxidizedmlx_amd import abi, nn
from oxidizedmlx_amd import backend as hb
from oxidizedmlx_amd.opkind import OpKind, meta
from oxidizedmlx_amd.tensor import Tensor, eval_all, value_and_grad

DTYPES = {"f32": (abi.F32, torch.float32), "bf16": (abi.BF16, torch.bfloat16), "f16": (abi.F16, torch.float16)}
EPS = 1e-5


def listed():
    return [
        # Matrix products (mlxhip_gemm). The smallest call: a product of a few
        # microseconds, where the launch counts.
        {"name": "gemm_f32_512", "kind": "gemm", "dtype": "f32", "ta": False, "tb": False,
         "m": 512, "n": 512, "k": 512, "batch": 1},
        # The large 16-bit product of a training step, C in the operands' dtype.
        {"name": "gemm_bf16_4096", "kind": "gemm", "dtype": "bf16", "ta": False, "tb": False,
         "m": 4096, "n": 4096, "k": 4096, "batch": 1},
        # Ragged sizes: rows that are no whole 16-byte chunks, edge tiles.
        {"name": "gemm_bf16_odd", "kind": "gemm", "dtype": "bf16", "ta": False, "tb": False,
         "m": 1000, "n": 777, "k": 1531, "batch": 1},
        # A Linear layer (x W^T) at decode time: eight rows against a whole
        # weight matrix, the up projection of the decoder's MLP.
        {"name": "linear_rows8", "kind": "gemm", "dtype": "f32", "ta": False, "tb": True,
         "m": 8, "n": 3072, "k": 768, "batch": 1},
        # A Linear layer in training: y = x W^T, dx = dy W, dW = dy^T x and the
        # bias gradient, at the transformer block's MLP sizes.
        {"name": "linear_train", "kind": "linear", "rows": 2048, "inputs": 1024, "outputs": 4096},
        # Softmax over a vocabulary, forward and gradient: long ragged rows.
        {"name": "softmax_vocab", "kind": "rows", "op": "softmax", "rows": 1000, "cols": 32003},
        # LayerNorm, forward and gradient, at the benchmark's size.
        {"name": "layernorm_4096", "kind": "rows", "op": "layernorm", "rows": 4096, "cols": 4096},
        # A mean over the last axis: a loss or a statistic per row.
        {"name": "reduce_last", "kind": "reduce", "op": "mean", "rows": 2048, "cols": 4096, "last": True},
        # Causal attention of 4 sequences x 16 heads, forward and gradient.
        {"name": "attention_train", "kind": "attention", "heads": 64, "tq": 512, "tk": 512, "dh": 64,
         "causal": True, "train": True},
        # The multi-head attention layer of one sequence (inference), built
        # and evaluated on a lazy stream.
        {"name": "mha_512", "kind": "mha", "seq": 512, "d_model": 1024, "heads": 16},
        # One training step of a transformer block: graph, autograd, every
        # gradient back to the caller.
        {"name": "block_train", "kind": "block", "batch": 4, "seq": 512, "d_model": 1024, "heads": 16,
         "fused": True},
        # The 12-layer decoder: a prompt, then greedy decoding, with logits.
        {"name": "generate", "kind": "generate", "layers": 12, "d_model": 768, "heads": 12, "vocab": 32000,
         "batch": 4, "prompt": 96, "new": 32},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """As _log, half of them rounded to a multiple of 64 where large."""
    n = _log(rng, lo, hi)
    return max(64, n // 64 * 64) if n >= 64 and rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choices(("gemm", "linear", "rows", "reduce", "attention", "mha", "block", "generate"),
                       (30, 10, 20, 10, 15, 5, 5, 5))[0]
    if kind == "gemm":
        while True:
            c = {"kind": "gemm", "dtype": rng.choice(("f32", "bf16", "f16")), "ta": rng.random() < 0.25,
                 "tb": rng.random() < 0.5, "m": _size(rng, 1, 4096), "n": _size(rng, 16, 4096),
                 "k": _size(rng, 32, 4096), "batch": rng.choice((1, 1, 1, 1, 4, 16, 32))}
            w = work(c)
            if w["flops"] <= 1.3e11 and w["bytes"] <= 4e8:
                return c
    if kind == "linear":
        return {"kind": "linear", "rows": _size(rng, 8, 4096), "inputs": _size(rng, 128, 4096),
                "outputs": _size(rng, 128, 4096)}
    if kind == "rows":
        while True:
            c = {"kind": "rows", "op": rng.choice(("softmax", "layernorm", "rmsnorm")),
                 "rows": _log(rng, 1, 16384), "cols": _size(rng, 16, 32768)}
            if c["rows"] * c["cols"] <= 1 << 25:
                return c
    if kind == "reduce":
        while True:
            c = {"kind": "reduce", "op": rng.choice(("sum", "mean", "max")), "rows": _size(rng, 8, 16384),
                 "cols": _size(rng, 8, 16384), "last": rng.random() < 0.5}
            if c["rows"] * c["cols"] <= 1 << 25:
                return c
    if kind == "attention":
        while True:
            train = rng.random() < 0.5
            t = 64 * _log(rng, 1, 32) if train else _log(rng, 16, 2048)
            c = {"kind": "attention", "heads": _log(rng, 1, 64), "tq": t, "tk": t,
                 "dh": 64 if train else rng.choice((32, 64, 128)), "causal": rng.random() < 0.75, "train": train}
            if not train and rng.random() < 0.3:  # a few new queries over a cache of keys
                c.update(tq=_log(rng, 1, 16), causal=False)
            if work(c)["flops"] <= 2.5e10:
                return c
    if kind == "mha":
        heads = rng.choice((4, 8, 12, 16))
        return {"kind": "mha", "seq": _log(rng, 16, 1024), "d_model": 64 * heads, "heads": heads}
    if kind == "block":
        heads = rng.choice((4, 8, 12, 16))
        return {"kind": "block", "batch": rng.randint(1, 4), "seq": 64 * rng.randint(1, 8), "d_model": 64 * heads,
                "heads": heads, "fused": rng.random() < 0.5}
    return {"kind": "generate", "layers": rng.choice((2, 4, 6)), "d_model": 768, "heads": 12, "vocab": 32000,
            "batch": rng.randint(1, 8), "prompt": _log(rng, 1, 96), "new": _log(rng, 1, 32)}


# ── inputs ────────────────────────────────────────────────────────────────

def _normal(gen, shape, std=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)


def _params(case, seed):
    """Inputs of a case as torch tensors on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "gemm":
        dt = DTYPES[case["dtype"]][1]
        m, n, k, b = case["m"], case["n"], case["k"], case["batch"]
        return {"a": _normal(g, (b, k, m) if case["ta"] else (b, m, k), dtype=dt),
                "b": _normal(g, (b, n, k) if case["tb"] else (b, k, n), dtype=dt)}
    if kind == "linear":
        r, i, o = case["rows"], case["inputs"], case["outputs"]
        return {"x": _normal(g, (r, i)), "w": _normal(g, (o, i), 0.02), "dy": _normal(g, (r, o))}
    if kind == "rows":
        shape = (case["rows"], case["cols"])
        return {"x": _normal(g, shape, 2.0), "dy": _normal(g, shape)}
    if kind == "reduce":
        return {"x": _normal(g, (case["rows"], case["cols"])) + 0.5}
    if kind == "attention":
        h, dh = case["heads"], case["dh"]
        p = {"q": _normal(g, (h, case["tq"], dh)), "k": _normal(g, (h, case["tk"], dh)),
             "v": _normal(g, (h, case["tk"], dh))}
        if case["train"]:
            p["do"] = _normal(g, (h, case["tq"], dh))
        return p
    if kind == "mha":
        d = case["d_model"]
        p = {"x": _normal(g, (case["seq"], d))}
        for nm in "qkvo":
            p["w" + nm] = _normal(g, (d, d), 0.02)
            p["b" + nm] = _normal(g, (d,), 0.02)
        return p
    if kind == "block":
        cfg = _block(case)
        p = {nm: _normal(g, shape, 0.02) for nm, shape in cfg.param_shapes().items()}
        p["x"] = _normal(g, (cfg.rows, cfg.d_model))
        p["gy"] = _normal(g, (cfg.rows, cfg.d_model))
        return p
    cfg = _decoder(case)
    d, v = cfg.d_model, cfg.vocab

    def weight(shape):  # the values that the bf16 decoder holds
        return _normal(g, shape, 0.02, torch.bfloat16).float()

    p = {"embedding": weight((v, d)), "lm_head": weight((v, d)),
         "layers": [{nm: weight(shape) for nm, shape in cfg.block(1, 1).param_shapes().items()}
                    for _ in range(cfg.n_layers)]}
    p["prompt"] = torch.randint(0, v, (case["batch"], case["prompt"]), generator=g, device="cuda").int()
    return p


def _block(case):
    return nn.BlockConfig(case["d_model"], case["heads"], case["seq"], case["batch"], eps=EPS,
                          fused_attention=case["fused"])


def _trained(cfg):
    """Every parameter but the keys' bias: it moves all of a row's scores by
    the same amount, so its gradient is zero and only rounding."""
    return [n for n in cfg.param_shapes() if n != "bk"]


def _decoder(case):
    return nn.DecoderConfig(n_layers=case["layers"], d_model=case["d_model"], n_heads=case["heads"],
                            vocab=case["vocab"], max_batch=case["batch"])


def prepare(case, seed):
    """Inputs, output buffers and what a program keeps: a lazy stream, a
    decoder with its weights loaded."""
    hb.init(0)
    p = _params(case, seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "gemm":
        s["c"] = torch.empty((case["batch"], case["m"], case["n"]), dtype=DTYPES[case["dtype"]][1], device="cuda")
    elif kind == "linear":
        s["y"], s["dx"], s["dw"] = (torch.empty_like(p[n]) for n in ("dy", "x", "w"))
        s["db"] = torch.empty(case["outputs"], device="cuda")
    elif kind == "rows":
        s["y"], s["dx"] = torch.empty_like(p["x"]), torch.empty_like(p["x"])
    elif kind == "reduce":
        s["y"] = torch.empty(case["rows"] if case["last"] else case["cols"], device="cuda")
    elif kind == "attention":
        s["o"] = torch.empty_like(p["q"])
        if case["train"]:
            s["dq"], s["dk"], s["dv"] = (torch.empty_like(p[n]) for n in "qkv")
    elif kind in ("mha", "block"):
        torch.cuda.synchronize()  # the lazy stream runs on a queue of its own
        s["stream"] = hb.HipStream()
    else:
        cfg = _decoder(case)
        dec = hb.HipDecoder(cfg)
        dec.load({"embedding": p["embedding"].cpu().numpy(), "lm_head": p["lm_head"].cpu().numpy(),
                  "layers": [{nm: t.cpu().numpy() for nm, t in lp.items()} for lp in p["layers"]]})
        return {"case": case, "decoder": dec, "prompt": p["prompt"].cpu().numpy()}
    s.update(p)
    return s


# ── one pass ──────────────────────────────────────────────────────────────

def _gemm_f32(ta, tb, m, n, k, a, b, c):
    hb.gemm(abi.F32, abi.F32, ta, tb, m, n, k, a.data_ptr(), a.shape[1], b.data_ptr(), b.shape[1], c.data_ptr(), n)


def _run_gemm(c, s):
    dt = DTYPES[c["dtype"]][0]
    m, n, k = c["m"], c["n"], c["k"]
    hb.gemm(dt, dt, c["ta"], c["tb"], m, n, k, s["a"].data_ptr(), m if c["ta"] else k,
            s["b"].data_ptr(), k if c["tb"] else n, s["c"].data_ptr(), n, batch=c["batch"],
            stride_a=m * k, stride_b=k * n, stride_c=m * n)
    return s["c"]


def _run_linear(c, s):
    r, i, o = c["rows"], c["inputs"], c["outputs"]
    _gemm_f32(False, True, r, o, i, s["x"], s["w"], s["y"])
    _gemm_f32(False, False, r, i, o, s["dy"], s["w"], s["dx"])
    _gemm_f32(True, False, o, i, r, s["dy"], s["x"], s["dw"])
    hb.eval_node_dev(OpKind.Sum(0), [(s["dy"].data_ptr(), (r, o))], meta([o]), s["db"].data_ptr())
    return {n: s[n] for n in ("y", "dx", "dw", "db")}


def _run_rows(c, s):
    r, n = c["rows"], c["cols"]
    x, dy, y, dx = (s[k].data_ptr() for k in ("x", "dy", "y", "dx"))
    if c["op"] == "softmax":
        hb.softmax_rows(x, y, r, n)
        hb.softmax_vjp_rows(dy, y, dx, r, n)
    elif c["op"] == "layernorm":
        hb.layernorm_rows(x, y, r, n, EPS)
        hb.layernorm_vjp_rows(dy, x, dx, r, n, EPS)
    else:
        hb.rmsnorm_rows(x, y, r, n, EPS)
        hb.rmsnorm_vjp_rows(dy, x, dx, r, n, EPS)
    return {"y": s["y"], "dx": s["dx"]}


def _run_reduce(c, s):
    axis = 1 if c["last"] else 0
    op = {"sum": OpKind.Sum, "mean": OpKind.Mean, "max": OpKind.Max}[c["op"]](axis)
    hb.eval_node_dev(op, [(s["x"].data_ptr(), (c["rows"], c["cols"]))], meta(s["y"].shape), s["y"].data_ptr())
    return s["y"]


def _run_attention(c, s):
    q, k, v, o = (s[n].data_ptr() for n in "qkvo")
    scale = 1.0 / math.sqrt(c["dh"])
    hb.attention(q, k, v, o, c["heads"], c["tq"], c["tk"], c["dh"], scale, c["causal"])
    if not c["train"]:
        return s["o"]
    hb.attention_vjp(q, k, v, o, s["do"].data_ptr(), s["dq"].data_ptr(), s["dk"].data_ptr(), s["dv"].data_ptr(),
                     c["heads"], c["tq"], c["dh"], scale, c["causal"])
    return {n: s[n] for n in ("o", "dq", "dk", "dv")}


def _run_mha(c, s):
    st = s["stream"]
    st.clear()
    t = {n: Tensor.view_device(v.data_ptr(), v.shape, st) for n, v in s.items() if isinstance(v, torch.Tensor)}
    layer = nn.MultiHeadAttention(*(nn.Linear(t["w" + n], t["b" + n]) for n in "qkvo"), c["heads"])
    return layer.forward_causal(t["x"]).to_numpy()


def _run_block(c, s):
    cfg, st = _block(c), s["stream"]
    st.clear()
    t = {n: Tensor.view_device(v.data_ptr(), v.shape, st) for n, v in s.items() if isinstance(v, torch.Tensor)}
    names = _trained(cfg)
    y = nn.TransformerBlock(cfg, {n: t[n] for n in cfg.param_shapes()})(t["x"])
    loss, grads = value_and_grad(y.mul(t["gy"]).sum_all(), [t[n] for n in names] + [t["x"]])
    eval_all([y, *grads])
    return {"y": y.to_numpy(), **{"d" + n: g.to_numpy() for n, g in zip(names + ["x"], grads)}}


def _run_generate(c, s):
    tokens, logits = s["decoder"].generate(s["prompt"], c["new"], logits=True)
    return {"tokens": tokens, "logits": logits}


RUN = {"gemm": _run_gemm, "linear": _run_linear, "rows": _run_rows, "reduce": _run_reduce,
       "attention": _run_attention, "mha": _run_mha, "block": _run_block, "generate": _run_generate}


def run(state):
    return RUN[state["case"]["kind"]](state["case"], state)


# ── what a pass cannot do without ─────────────────────────────────────────

def _pairs(c):
    """(query, visible key) pairs of one head."""
    if not c["causal"]:
        return c["tq"] * c["tk"]
    return sum(min(i + 1, c["tk"]) for i in range(c["tq"]))


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemm":
        m, n, k, b = c["m"], c["n"], c["k"], c["batch"]
        size = 4 if c["dtype"] == "f32" else 2
        return {"bytes": b * (m * k + k * n + m * n) * size, "flops": 2 * b * m * n * k}
    if kind == "linear":
        r, i, o = c["rows"], c["inputs"], c["outputs"]
        return {"bytes": 4 * (2 * r * i + 2 * o * i + 2 * r * o + o), "flops": 6 * r * i * o}
    if kind == "rows":
        return {"bytes": 16 * c["rows"] * c["cols"], "flops": 0}
    if kind == "reduce":
        return {"bytes": 4 * (c["rows"] * c["cols"] + (c["rows"] if c["last"] else c["cols"])), "flops": 0}
    if kind == "attention":
        q, k = c["heads"] * c["tq"] * c["dh"], c["heads"] * c["tk"] * c["dh"]
        n = c["heads"] * _pairs(c) * c["dh"]
        return {"bytes": 4 * (5 * q + 5 * k if c["train"] else 2 * q + 2 * k), "flops": n * (14 if c["train"] else 4)}
    if kind == "mha":
        s, d = c["seq"], c["d_model"]
        return {"bytes": 4 * (4 * d * d + 2 * s * d), "flops": 8 * s * d * d + 4 * d * (s * (s + 1) // 2)}
    if kind == "block":
        cfg = _block(c)
        weights = sum(math.prod(s) for s in cfg.param_shapes().values())
        return {"bytes": 4 * (2 * weights + 4 * cfg.rows * cfg.d_model), "flops": 3 * cfg.forward_flops()}
    cfg = _decoder(c)
    # The weights once for the prompt and once per further token; the logits
    # and every layer's K and V rows written.
    b, p, n = c["batch"], c["prompt"], c["new"]
    steps = p + n - 1
    return {"bytes": n * cfg.step_weight_bytes() + 4 * b * steps * (cfg.vocab + 2 * cfg.d_model * cfg.n_layers),
            "flops": b * steps * cfg.step_weight_bytes()}


def tolerance(case):
    """About four times what the paths showed against exact(): C rounded to 8
    or 11 significant bits 1.7e-3 and 2.1e-4, f32 sums up to 9e-7 in a layer,
    4e-6 in a block's gradients, 4e-7 in the decoder's logits."""
    kind = case["kind"]
    if kind == "gemm" and case["dtype"] != "f32":
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 1e-3}
    if kind == "generate":
        return {"rel": 4e-6, "differ": 0.01}  # an equal pair of logits may give the other token
    return {"rel": 1.5e-5 if kind == "block" else 4e-6}


# ── the same in 64 bits, by torch alone ───────────────────────────────────

def _attend(q, k, v, scale, causal):
    s = torch.matmul(q, k.transpose(-1, -2)) * scale
    if causal:
        s = s.masked_fill(torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1), -math.inf)
    return torch.matmul(torch.softmax(s, -1), v)


def _rms(x):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS)


def _split(x, batch, heads):
    """[batch * t, d] -> [batch, heads, t, d / heads]."""
    return x.reshape(batch, -1, heads, x.shape[-1] // heads).transpose(1, 2)


def _merge(x):
    b, h, t, dh = x.shape
    return x.transpose(1, 2).reshape(b * t, h * dh)


def _exact_attention(c, p):
    outs = []
    for i in range(c["heads"]):  # head by head: bounded memory
        q, k, v = (p[n][i].requires_grad_(c["train"]) for n in "qkv")
        o = _attend(q, k, v, 1.0 / math.sqrt(c["dh"]), c["causal"])
        outs.append((o.detach(), *(torch.autograd.grad(o, (q, k, v), p["do"][i]) if c["train"] else ())))
    outs = [torch.stack(t) for t in zip(*outs)]
    return dict(zip(("o", "dq", "dk", "dv"), outs)) if c["train"] else outs[0]


def _exact_block(c, p):
    names = _trained(_block(c))
    t = {n: p[n].requires_grad_() for n in (*_block(c).param_shapes(), "x")}
    b, h = c["batch"], c["heads"]
    x = t["x"]
    a = _rms(x)
    q, k, v = (_split(a @ t["w" + n].T + t["b" + n], b, h) for n in "qkv")
    o = _attend(q, k, v, 1.0 / math.sqrt(c["d_model"] // h), True)
    hid = x + (_merge(o) @ t["wo"].T + t["bo"])
    y = hid + (torch.nn.functional.silu(_rms(hid) @ t["w1"].T + t["b1"]) @ t["w2"].T + t["b2"])
    grads = torch.autograd.grad(y, [t[n] for n in names + ["x"]], p["gy"])
    return {"y": y.detach(), **{"d" + n: g for n, g in zip(names + ["x"], grads)}}


def _exact_generate(c, p):
    """Logits of every position; the tokens fed back are the 64-bit argmax."""
    b, heads = c["batch"], c["heads"]
    scale = 1.0 / math.sqrt(c["d_model"] // heads)
    keys, values = [None] * c["layers"], [None] * c["layers"]
    tokens, logits = p["prompt"].long(), []
    for step in range(c["new"]):
        x = p["embedding"][tokens].reshape(-1, c["d_model"])
        for i, w in enumerate(p["layers"]):
            a = _rms(x)
            q, k, v = (_split(a @ w["w" + n].T + w["b" + n], b, heads) for n in "qkv")
            keys[i] = k if step == 0 else torch.cat([keys[i], k], 2)
            values[i] = v if step == 0 else torch.cat([values[i], v], 2)
            x = x + (_merge(_attend(q, keys[i], values[i], scale, step == 0)) @ w["wo"].T + w["bo"])
            x = x + (torch.nn.functional.silu(_rms(x) @ w["w1"].T + w["b1"]) @ w["w2"].T + w["b2"])
        logits.append((_rms(x) @ p["lm_head"].T).reshape(b, -1, c["vocab"]))
        tokens = logits[-1][:, -1:].argmax(-1)
    return {"tokens": None, "logits": torch.cat(logits, 1)}


def exact(case, seed):
    c, kind = case, case["kind"]

    def wide(v):
        if isinstance(v, dict):
            return {k: wide(x) for k, x in v.items()}
        return [wide(x) for x in v] if isinstance(v, list) else v.double()

    p = wide(_params(case, seed))
    if kind == "gemm":
        return torch.matmul(p["a"].transpose(1, 2) if c["ta"] else p["a"], p["b"].transpose(1, 2) if c["tb"] else p["b"])
    if kind == "linear":
        return {"y": p["x"] @ p["w"].T, "dx": p["dy"] @ p["w"], "dw": p["dy"].T @ p["x"], "db": p["dy"].sum(0)}
    if kind == "rows":
        x = p["x"].requires_grad_()
        if c["op"] == "softmax":
            y = torch.softmax(x, -1)
        elif c["op"] == "layernorm":
            y = torch.nn.functional.layer_norm(x, x.shape[-1:], eps=EPS)
        else:
            y = _rms(x)
        return {"y": y.detach(), "dx": torch.autograd.grad(y, x, p["dy"])[0]}
    if kind == "reduce":
        axis = 1 if c["last"] else 0
        return p["x"].amax(axis) if c["op"] == "max" else getattr(p["x"], c["op"])(axis)
    if kind == "attention":
        return _exact_attention(c, p)
    if kind == "mha":
        q, k, v = (_split(p["x"] @ p["w" + n].T + p["b" + n], 1, c["heads"]) for n in "qkv")
        o = _attend(q, k, v, 1.0 / math.sqrt(c["d_model"] // c["heads"]), True)
        return _merge(o) @ p["wo"].T + p["bo"]
    return (_exact_block if kind == "block" else _exact_generate)(c, p)
