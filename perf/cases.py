"""The work that programs have this framework do, as cases that can be timed and compared.

Every case goes through the public entry points: the C ABI of include/midman_hip.h with caller-owned device buffers
(the way the header describes and a Rust binding uses it) and, for whole models, the Python mirror's Model. Inputs
come from a seed, with the distributions of the configurations: activations ~ N(0, 1), weights ~ N(0, 0.02), token
ids uniform over the vocabulary. Everything is f32, as the framework is.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "midman-ai_amd"))
import midman_hip as mh  # noqa: E402

STD = 0.02
EPS = 1e-5
THETA = 10000.0
# vocab, d_model, layers, heads, kv_heads, d_ff, max_seq: the presets' dimensions
TINY = dict(vocab=4096, d=128, layers=4, heads=4, kv=4, ff=344, max_seq=256)
LARGE = dict(vocab=32000, d=2048, layers=20, heads=16, kv=8, ff=5632, max_seq=2048)


def listed():
    return [
        # one projection of the smallest preset, 2 x 32 tokens: a call that is all latency
        dict(name="gemm_smoke", kind="gemm", form="nn", m=64, k=64, n=176, accumulate=False),
        # gradients added up over a batch whose token count and widths are no multiple of anything
        dict(name="gemm_ragged", kind="gemm", form="tn", m=1003, k=1517, n=770, accumulate=True),
        # a linear layer's training share, forward and both gradients, at 8 x 256 tokens
        dict(name="linear_train", kind="linear", rows=2048, k=1024, n=4096),
        # the tied head of the large preset at 4 x 1024 tokens: logits over 32000 words
        dict(name="head", kind="gemm", form="nt", m=4096, k=2048, n=32000, accumulate=False),
        # the MLP's backward at d_model 1024, 2 x 1024 tokens
        dict(name="swiglu_bwd", kind="swiglu_bwd", rows=2048, d=1024, ff=2816),
        # one decoder block alone, grouped heads, at 8 x 1024 tokens
        dict(name="block", kind="block", b=8, t=1024, d=1024, h=16, hkv=8, ff=2816),
        # attention of the large preset's layer, 4 x 1024 tokens
        dict(name="attn", kind="attn", b=4, h=16, hkv=8, t=1024, hd=128),
        # attention's gradients with heads of 64 and a ragged sequence
        dict(name="attn_bwd", kind="attn_bwd", b=4, h=12, hkv=12, t=1000, hd=64),
        # the norm before each block and its gradients, 4 x 1024 tokens
        dict(name="norm_train", kind="norm", rows=4096, d=2048),
        # evaluation of the tiny preset at its training batch: the loss of 8 x 256 new tokens
        dict(name="tiny_loss", kind="loss", b=8, t=256, **TINY),
        # its training: loss and every gradient, read back
        dict(name="tiny_train", kind="train", b=8, t=256, **TINY),
        # evaluation of the large preset, 4 x 1024 tokens
        dict(name="large_loss", kind="loss", b=4, t=1024, **LARGE),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size in [lo, hi], spread over its logarithm: half of them multiples of 64 where there is room, the others as they fall."""
    v = _log(rng, lo, hi)
    return max(64, v // 64 * 64) if v >= 128 and rng.random() < 0.5 else v


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "linear", "swiglu_bwd", "block", "attn", "attn_bwd", "norm", "loss", "train"])
    if kind in ("gemm", "linear"):
        while True:
            m, k, n = _size(rng, 32, 8192), _size(rng, 32, 8192), _size(rng, 32, 32000)
            if m * k * n <= 4096 * 2048 * 16000:
                break
        if kind == "linear":
            return dict(kind=kind, rows=m, k=k, n=n)
        return dict(kind=kind, form=rng.choice(["nn", "nt", "tn"]), m=m, k=k, n=n, accumulate=rng.random() < 0.25)
    if kind == "swiglu_bwd":
        return dict(kind=kind, rows=_size(rng, 64, 8192), d=_size(rng, 64, 2048), ff=4 * _size(rng, 44, 1408))
    if kind == "norm":
        return dict(kind=kind, rows=_size(rng, 64, 16384), d=_size(rng, 64, 4096))
    if kind in ("loss", "train"):
        hd, heads = rng.choice([(16, 4), (32, 4), (64, 6), (64, 12)])
        d, t = hd * heads, _log(rng, 24, 512)
        kv = rng.choice([heads, heads // 2])
        return dict(kind=kind, b=_log(rng, 1, max(2, 4096 // t)), t=t, vocab=_log(rng, 256, 8192), d=d,
                    layers=rng.randint(1, 6), heads=heads, kv=kv, ff=8 * round(d / 3), max_seq=512)
    hd = rng.choice([16, 32, 64, 128])
    h = rng.choice([4, 6, 8, 12, 16])
    hkv = rng.choice([h, h // 2])
    t = _size(rng, 24, 2048)
    b = _log(rng, 1, max(2, 8192 // t))
    if kind == "block":
        return dict(kind=kind, b=b, t=t, d=h * hd, h=h, hkv=hkv, ff=8 * round(h * hd / 3))
    return dict(kind=kind, b=b, h=h, hkv=hkv, t=t, hd=hd)


# ---- inputs --------------------------------------------------------------------

_context = None


def _ctx():
    """The program's one context."""
    global _context
    if _context is None:
        _context = mh.Context(0)
    return _context


class _Cuda:
    """A DeviceArray's memory, for torch."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = dict(shape=array.shape, typestr="<f4", data=(array.ptr, False), version=2)


def _view(array):
    return torch.as_tensor(_Cuda(array), device="cuda")


def _randn(seed, shapes):
    """f32 normals on the GPU for {name: (shape, std)}, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return {n: torch.randn(s, generator=g, device="cuda") * std for n, (s, std) in shapes.items()}


def _inputs(c):
    """{name: (shape, std)} of a case's random arrays."""
    kind = c["kind"]
    if kind == "gemm":
        m, k, n, f = c["m"], c["k"], c["n"], c["form"]
        s = {"a": ((k, m) if f == "tn" else (m, k), 1.0), "b": ((n, k) if f == "nt" else (k, n), STD)}
        if c["accumulate"]:
            s["c"] = ((m, n), 1.0)
        return s
    if kind == "linear":
        r, k, n = c["rows"], c["k"], c["n"]
        return {"a": ((r, k), 1.0), "b": ((k, n), STD), "dc": ((r, n), 1.0)}
    if kind == "swiglu_bwd":
        r, d, ff = c["rows"], c["d"], c["ff"]
        return {"x": ((r, d), 1.0), "wg": ((d, ff), STD), "wu": ((d, ff), STD), "wd": ((ff, d), STD), "dout": ((r, d), 1.0)}
    if kind == "block":
        d, ff, kv = c["d"], c["ff"], c["hkv"] * (c["d"] // c["h"])
        return {"x": ((c["b"], c["t"], d), 1.0), "q": ((d, d), STD), "k": ((d, kv), STD), "v": ((d, kv), STD), "o": ((d, d), STD),
                "gate": ((d, ff), STD), "up": ((d, ff), STD), "down": ((ff, d), STD)}
    if kind in ("attn", "attn_bwd"):
        q, kv = (c["b"], c["h"], c["t"], c["hd"]), (c["b"], c["hkv"], c["t"], c["hd"])
        s = {"q": (q, 1.0), "k": (kv, 1.0), "v": (kv, 1.0)}
        if kind == "attn_bwd":
            s["dout"] = (q, 1.0)
        return s
    return {"x": ((c["rows"], c["d"]), 1.0), "w": ((c["d"],), 0.1), "dy": ((c["rows"], c["d"]), 1.0)}  # norm; w moved to 1 + w


def _drawn(c, seed):
    t = _randn(seed, _inputs(c))
    if c["kind"] == "norm":
        t["w"] += 1.0
    return t


def _model_weights(c, seed):
    """The parameters in the reference order, as the seeded init distributes them."""
    d, ff, kv, out = c["d"], c["ff"], c["kv"] * (c["d"] // c["heads"]), STD / math.sqrt(2 * c["layers"])
    shapes = [("embed", (c["vocab"], d), STD)]
    for i in range(c["layers"]):
        p = "%d." % i
        shapes += [(p + "attn_norm", (d,), 0.0), (p + "q", (d, d), STD), (p + "k", (d, kv), STD), (p + "v", (d, kv), STD),
                   (p + "o", (d, d), out), (p + "mlp_norm", (d,), 0.0), (p + "gate", (d, ff), STD), (p + "up", (d, ff), STD),
                   (p + "down", (ff, d), out)]
    shapes.append(("final_norm", (d,), 0.0))
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    w = torch.empty(sum(math.prod(s) for _, s, _ in shapes), device="cuda")
    parts, at = {}, 0
    for name, s, std in shapes:
        v = w[at:at + math.prod(s)].view(s)
        v.fill_(1.0) if std == 0.0 else v.normal_(0.0, std, generator=g)
        parts[name] = v
        at += v.numel()
    ids = torch.randint(0, c["vocab"], (c["b"], c["t"] + 1), generator=g, device="cuda")
    return w, parts, ids


class _State(dict):
    def __del__(self):
        if "model" in self:
            self["model"].close()


def prepare(case, seed):
    c, ctx = case, _ctx()
    s = _State(case=c)
    if c["kind"] in ("loss", "train"):
        w, _, ids = _model_weights(c, seed)
        config = [c["vocab"], c["d"], c["layers"], c["heads"], c["kv"], c["ff"], c["max_seq"], THETA, EPS, 1]
        s["model"] = mh.Model.from_weights(ctx, config, w.cpu().numpy())
        ids = ids.cpu().numpy().astype(np.int32)
        s["x"], s["y"] = np.ascontiguousarray(ids[:, :-1]).reshape(-1), np.ascontiguousarray(ids[:, 1:]).reshape(-1)
        return s
    t = _drawn(c, seed)
    if c["kind"] == "block":
        one = torch.ones(c["d"], device="cuda")
        flat = [one] + [t[n].reshape(-1) for n in ("q", "k", "v", "o")] + [one] + [t[n].reshape(-1) for n in ("gate", "up", "down")]
        t = {"x": t["x"], "weights": torch.cat(flat)}
        s["tables"] = mh.RotaryTables(ctx, c["d"] // c["h"], c["t"], THETA)
    for name, v in t.items():
        s[name] = ctx.empty(tuple(v.shape))
        _view(s[name]).copy_(v)
    shape = lambda name: s[name].shape  # noqa: E731
    outs = {
        "gemm": lambda: {} if c["accumulate"] else {"c": (c["m"], c["n"])},
        "linear": lambda: {"c": (c["rows"], c["n"]), "da": shape("a"), "db": shape("b")},
        "swiglu_bwd": lambda: {"dx": shape("x"), "dwg": shape("wg"), "dwu": shape("wu"), "dwd": shape("wd")},
        "block": lambda: {"out": shape("x")},
        "attn": lambda: {"out": shape("q")},
        "attn_bwd": lambda: {"dq": shape("q"), "dk": shape("k"), "dv": shape("v")},
        "norm": lambda: {"y": shape("x"), "dx": shape("x"), "dw": shape("w")},
    }[c["kind"]]()
    for name, sh in outs.items():
        s[name] = ctx.empty(sh)
    if c["kind"] == "gemm":
        outs = {"c": None}
    s["outs"] = {name: _view(s[name]) for name in outs}
    torch.cuda.synchronize()  # the inputs are there before the context's own stream reads them
    return s


# ---- one pass ------------------------------------------------------------------

def _call(name, *args):
    """One entry point of the C ABI, with DeviceArrays for its pointers."""
    mh.check(getattr(mh.lib(), name)(_ctx().handle, *[a.ptr if isinstance(a, mh.DeviceArray) else a for a in args]))


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "loss":
        return {"loss": s["model"].loss(s["x"], s["y"], c["b"], c["t"])}
    if kind == "train":
        loss = s["model"].backward(s["x"], s["y"], c["b"], c["t"])
        return {"loss": loss, "grads": s["model"].grads()}
    if kind == "gemm":
        _call("mmh_gemm_" + c["form"], s["a"], s["b"], s["c"], c["m"], c["k"], c["n"], 1 if c["accumulate"] else 0)
    elif kind == "linear":
        _call("mmh_gemm_nn", s["a"], s["b"], s["c"], c["rows"], c["k"], c["n"], 0)
        _call("mmh_matmul_backward", s["a"], s["b"], s["dc"], s["da"], s["db"], c["rows"], c["k"], c["n"])
    elif kind == "swiglu_bwd":
        _call("mmh_swiglu_backward", s["x"], s["wg"], s["wu"], s["wd"], s["dout"], c["rows"], c["d"], c["ff"],
              s["dx"], s["dwg"], s["dwu"], s["dwd"])
    elif kind == "block":
        _call("mmh_block_forward", s["x"], s["weights"], s["tables"].cos, s["tables"].sin, c["b"], c["t"], c["d"], c["h"],
              c["hkv"], c["ff"], EPS, s["out"])
    elif kind == "attn":
        _call("mmh_causal_attention", s["q"], s["k"], s["v"], c["b"], c["h"], c["hkv"], c["t"], c["hd"], s["out"])
    elif kind == "attn_bwd":
        _call("mmh_causal_attention_backward", s["q"], s["k"], s["v"], s["dout"], c["b"], c["h"], c["hkv"], c["t"], c["hd"],
              s["dq"], s["dk"], s["dv"])
    else:
        _call("mmh_rms_norm", s["x"], s["w"], c["rows"], c["d"], EPS, s["y"])
        _call("mmh_rms_norm_backward", s["x"], s["w"], s["dy"], c["rows"], c["d"], EPS, s["dx"], s["dw"])
    return s["outs"]


# ---- what a pass cannot do without -----------------------------------------------

def work(case):
    c = case
    kind = c["kind"]
    if kind == "gemm":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": 4.0 * (m * k + k * n + m * n * (2 if c["accumulate"] else 1)), "flops": 2.0 * m * k * n}
    if kind == "linear":
        m, k, n = c["rows"], c["k"], c["n"]
        return {"bytes": 4.0 * (2 * m * k + 2 * k * n + 2 * m * n), "flops": 6.0 * m * k * n}
    if kind == "swiglu_bwd":  # gate and up again, then the gradients of three products
        m, d, ff = c["rows"], c["d"], c["ff"]
        return {"bytes": 4.0 * (3 * m * d + 6 * d * ff), "flops": 2.0 * m * d * ff * 8}
    if kind == "block":
        rows, d, ff, kv = c["b"] * c["t"], c["d"], c["ff"], c["hkv"] * (c["d"] // c["h"])
        w = 2 * d * d + 2 * d * kv + 3 * d * ff
        return {"bytes": 4.0 * (2 * rows * d + w), "flops": 2.0 * rows * w + 2.0 * c["b"] * d * c["t"] * (c["t"] + 1)}
    if kind in ("attn", "attn_bwd"):
        q, kv = c["b"] * c["h"] * c["t"] * c["hd"], c["b"] * c["hkv"] * c["t"] * c["hd"]
        f = 2.0 * q * (c["t"] + 1)
        # the backward forms the scores again and four products from them
        return {"bytes": 4.0 * (2 * q + 2 * kv), "flops": f} if kind == "attn" else {"bytes": 4.0 * (3 * q + 4 * kv), "flops": 2.5 * f}
    if kind == "norm":
        return {"bytes": 4.0 * (4 * c["rows"] * c["d"] + 2 * c["d"]), "flops": 14.0 * c["rows"] * c["d"]}
    rows, d, ff, kv, L = c["b"] * c["t"], c["d"], c["ff"], c["kv"] * (c["d"] // c["heads"]), c["layers"]
    w = L * (2 * d * d + 2 * d * kv + 3 * d * ff) + c["vocab"] * d
    f = 2.0 * rows * w + 2.0 * L * c["b"] * d * c["t"] * (c["t"] + 1)
    return {"bytes": 4.0 * w, "flops": f} if kind == "loss" else {"bytes": 8.0 * w, "flops": 3 * f}


def tolerance(case):
    # f32 sums of up to 8192 terms are 1e-6 from the 64-bit result (2e-6 at the longest), a mean loss over thousands of
    # tokens within its own rounding
    return {"rel": 1e-6} if case["kind"] == "loss" else {"rel": 1e-5}


# ---- the same in 64 bits -----------------------------------------------------------

def _rms(x, w):
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * w


def _rotate(x):
    """x [b, h, t, hd] at positions 0..t-1, with the tables' f32 values."""
    t, half = x.shape[-2], x.shape[-1] // 2
    angle = np.outer(np.arange(t, dtype=np.float64), THETA ** (-np.arange(half, dtype=np.float64) / half))
    cos, sin = (torch.from_numpy(f(angle).astype(np.float32)).double().to(x.device) for f in (np.cos, np.sin))
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _attend(q, k, v):
    h, t = q.shape[1], q.shape[2]
    k, v = (x.repeat_interleave(h // x.shape[1], 1) for x in (k, v))
    mask = torch.ones(t, t, dtype=torch.bool, device=q.device).tril()
    out = []
    for i in range(q.shape[0]):  # a sequence at a time: the scores are [h, t, t]
        s = (q[i] @ k[i].transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
        out.append(torch.softmax(s.masked_fill(~mask, -math.inf), -1) @ v[i])
    return torch.stack(out)


def _block(x, w, h, hkv):
    b, t, d = x.shape
    heads = lambda y, n: _rotate(y.view(b, t, n, d // h).transpose(1, 2))  # noqa: E731
    y = _rms(x, w["attn_norm"])
    v = (y @ w["v"]).view(b, t, hkv, d // h).transpose(1, 2)
    x = x + _attend(heads(y @ w["q"], h), heads(y @ w["k"], hkv), v).transpose(1, 2).reshape(b, t, d) @ w["o"]
    y = _rms(x, w["mlp_norm"])
    return x + (torch.nn.functional.silu(y @ w["gate"]) * (y @ w["up"])) @ w["down"]


def _model_loss(c, w, ids):
    x = w["embed"][ids[:, :-1]]
    for i in range(c["layers"]):
        p = "%d." % i
        x = _block(x, {n[len(p):]: v.double() for n, v in w.items() if n.startswith(p)}, c["heads"], c["kv"])
    x = _rms(x, w["final_norm"]).reshape(-1, c["d"])
    y = ids[:, 1:].reshape(-1)
    total = 0.0
    for at in range(0, len(y), 1024):  # some rows of logits at a time
        z = x[at:at + 1024] @ w["embed"].T
        total = total + torch.nn.functional.cross_entropy(z, y[at:at + 1024], reduction="sum")
    return total / len(y)


def _grads(f, *args):
    args = [a.requires_grad_() for a in args]
    out, dout = f(*args)
    return torch.autograd.grad(out, args, dout)


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind in ("loss", "train"):
        flat, parts, ids = _model_weights(c, seed)
        if kind == "loss":
            with torch.no_grad():
                w = {n: v.double() if "." not in n else v for n, v in parts.items()}
                return {"loss": float(_model_loss(c, w, ids))}
        w = {n: v.double().requires_grad_() for n, v in parts.items()}
        loss = _model_loss(c, w, ids)
        grads = torch.autograd.grad(loss, list(w.values()))
        return {"loss": float(loss), "grads": torch.cat([g.reshape(-1) for g in grads])}
    t = {n: v.double() for n, v in _drawn(c, seed).items()}
    if kind == "gemm":
        a, b = t["a"].T if c["form"] == "tn" else t["a"], t["b"].T if c["form"] == "nt" else t["b"]
        # an accumulated product depends on how many were added: its first pass
        return {"c": a @ b + t["c"] if c["accumulate"] else a @ b}
    if kind == "linear":
        return {"c": t["a"] @ t["b"], "da": t["dc"] @ t["b"].T, "db": t["a"].T @ t["dc"]}
    if kind == "swiglu_bwd":
        f = lambda x, g, u, d: ((torch.nn.functional.silu(x @ g) * (x @ u)) @ d, t["dout"])  # noqa: E731
        return dict(zip(("dx", "dwg", "dwu", "dwd"), _grads(f, t["x"], t["wg"], t["wu"], t["wd"])))
    if kind == "block":
        t["attn_norm"] = t["mlp_norm"] = torch.ones(c["d"], dtype=torch.float64, device="cuda")
        return {"out": _block(t["x"], t, c["h"], c["hkv"])}
    if kind == "attn":
        return {"out": _attend(t["q"], t["k"], t["v"])}
    if kind == "attn_bwd":
        return dict(zip(("dq", "dk", "dv"), _grads(lambda q, k, v: (_attend(q, k, v), t["dout"]), t["q"], t["k"], t["v"])))
    dx, dw = _grads(lambda x, w: (_rms(x, w), t["dy"]), t["x"], t["w"])
    return {"y": _rms(t["x"], t["w"]).detach(), "dx": dx, "dw": dw}
