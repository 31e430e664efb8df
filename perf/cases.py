"""The work that programs built on this backend have it do, as measurable cases.

Every case goes through the public entry points of ``zigneuron_amd``: the
device-pointer calls of ``Context`` (tensors resident in HBM, the form a
training loop or a server uses) and, for one family, the host-slice calls of
``Backend`` (the reference's own call form).  Everything is float32.

Families (``kind``) and what each stands for:
  gemm       one ``Context.sgemm`` in any of the three layouts, plain, with a
             fused bias + activation or accumulating: an inference layer of a
             few rows, the square products, ragged matrices, the largest ones;
  batched    one ``Context.sgemm_strided_batched``: the score and value
             products of multi-head attention run as GEMMs;
  mlp        one training step of a two-layer perceptron (both forwards, both
             backwards), the smallest launches;
  dense      one training step of a single Dense layer: fused forward, then
             activation derivative, input, weight and bias gradients;
  attention  fused softmax attention over a batch of heads, or one head;
  conv       a convolution's forward and backward, in the two weight orders of
             the reference (im2col order and OIHW);
  host       one ``Backend.matMulBias*`` call on host arrays.
"""
import math

import numpy as np
import torch

from zigneuron_amd import Backend, Context

ACTS = ("linear", "relu", "sigmoid", "tanh")
_handles = {}


def _ctx():
    """The device context a program creates once and keeps."""
    if "ctx" not in _handles:
        _handles["ctx"] = Context(0)
    return _handles["ctx"]


def _backend():
    if "backend" not in _handles:
        _handles["backend"] = Backend.init(0)
    return _handles["backend"]


# ------------------------------------------------------------------ the cases
def _gemm(layout, m, n, k, act="linear", bias=False, accumulate=False):
    return {"kind": "gemm", "layout": layout, "m": m, "n": n, "k": k, "act": act, "bias": bias, "accumulate": accumulate}


def _conv(order, batch, c, oc, hw, ker, stride, pad):
    return {"kind": "conv", "order": order, "batch": batch, "c": c, "oc": oc, "h": hw, "w": hw, "ker": ker,
            "stride": stride, "pad": pad}


def listed():
    return [
        # training step of the 784-128-10 classifier, batch 256
        {"name": "mlp_step", "kind": "mlp", "batch": 256, "inp": 784, "hidden": 128, "out": 10, "act": "relu"},
        # a served Dense layer: 8 requests through 1024 x 1024 weights, bias and sigmoid fused
        {"name": "dense_serve", **_gemm("nn", 8, 1024, 1024, "sigmoid", True)},
        # a square product of ordinary size
        {"name": "gemm_512", **_gemm("nn", 512, 512, 512)},
        # a ragged product: no extent is a multiple of 4
        {"name": "gemm_ragged", **_gemm("nn", 4097, 1023, 777)},
        # the largest single product
        {"name": "gemm_8192", **_gemm("nn", 8192, 8192, 8192)},
        # training step of a 1024 x 1024 Dense layer on 4096 rows: NN, NT and TN products
        {"name": "dense_step", "kind": "dense", "batch": 4096, "inp": 1024, "out": 1024, "act": "tanh"},
        # the score products of 128 heads of 1024 positions and 64 dimensions
        {"name": "scores", "kind": "batched", "layout": "nt", "m": 1024, "n": 1024, "k": 64, "batch": 128},
        # the whole attention of those heads
        {"name": "attention", "kind": "attention", "batch": 128, "seq": 1024, "dim": 64},
        # one head at a time, as the reference's attentionForward takes it: a ragged length and head dimension
        {"name": "attention_head", "kind": "attention", "batch": 1, "seq": 1000, "dim": 80},
        # training step of a middle convolution layer: 64 -> 128 channels, 3x3, 56 x 56, batch 32
        {"name": "conv_step", **_conv("im2col", 32, 64, 128, 56, 3, 1, 1)},
        # training step of a first convolution layer: 3 colour channels, OIHW weights, stride 2
        {"name": "conv_first", **_conv("direct", 16, 3, 32, 64, 5, 2, 2)},
        # the reference's call form on host arrays: one hidden layer of the classifier
        {"name": "host_dense", "kind": "host", "m": 256, "n": 128, "k": 784, "act": "relu"},
    ]


def _log(rng, lo, hi):
    """An integer spread over [lo, hi] on a logarithmic scale."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("gemm", "gemm", "gemm", "batched", "mlp", "dense", "attention", "attention", "conv", "conv", "host"))
    if kind == "gemm":
        mode = rng.choice(("plain", "plain", "bias", "accumulate"))
        return _gemm(rng.choice(("nn", "nt", "tn")), _log(rng, 1, 8192), _log(rng, 10, 8192), _log(rng, 16, 8192),
                     rng.choice(ACTS) if mode == "bias" else "linear", mode == "bias", mode == "accumulate")
    if kind == "batched":
        return {"kind": "batched", "layout": rng.choice(("nn", "nt", "tn")), "m": _log(rng, 32, 1024),
                "n": _log(rng, 32, 1024), "k": _log(rng, 16, 1024), "batch": _log(rng, 4, 128)}
    if kind == "mlp":
        # no relu here or below where a backward follows: a unit within a rounding of zero would switch its whole gradient
        return {"kind": "mlp", "batch": _log(rng, 8, 1024), "inp": _log(rng, 16, 1024), "hidden": _log(rng, 16, 512),
                "out": _log(rng, 2, 16), "act": rng.choice(("sigmoid", "tanh"))}
    if kind == "dense":
        return {"kind": "dense", "batch": _log(rng, 16, 4096), "inp": _log(rng, 64, 4096), "out": _log(rng, 64, 4096),
                "act": rng.choice(("linear", "sigmoid", "tanh"))}
    if kind == "attention":
        return {"kind": "attention", "batch": _log(rng, 1, 128), "seq": _log(rng, 16, 2048), "dim": _log(rng, 16, 128)}
    if kind == "conv":
        while True:
            ker = rng.choice((1, 3, 3, 3, 5))
            c = _conv(rng.choice(("im2col", "direct")), _log(rng, 1, 32), _log(rng, 1, 128), _log(rng, 8, 128),
                      _log(rng, 8, 64), ker, rng.choice((1, 1, 2)), rng.choice((0, ker // 2)))
            if work(c)["flops"] <= 2.5e10:
                return c
    return {"kind": "host", "m": _log(rng, 1, 512), "n": _log(rng, 10, 1024), "k": _log(rng, 16, 1024),
            "act": rng.choice(ACTS)}


def _out_hw(c):
    return tuple((c[x] + 2 * c["pad"] - c["ker"]) // c["stride"] + 1 for x in ("h", "w"))


def work(case):
    c, kind = case, case["kind"]
    if kind in ("gemm", "host"):
        m, n, k = c["m"], c["n"], c["k"]
        extra = (n if c.get("bias", kind == "host") else 0) + (m * n if c.get("accumulate") else 0)
        return {"bytes": 4 * (m * k + k * n + m * n + extra), "flops": 2 * m * n * k}
    if kind == "batched":
        m, n, k, b = c["m"], c["n"], c["k"], c["batch"]
        return {"bytes": 4 * b * (m * k + k * n + m * n), "flops": 2 * b * m * n * k}
    if kind == "mlp":
        b, i, h, o = c["batch"], c["inp"], c["hidden"], c["out"]
        # read x, both weights and biases, grad_y; write h, y, gaa1, gaa2, grad_x, grad_h and the four parameter gradients
        return {"bytes": 4 * (2 * b * i + 3 * b * h + 3 * b * o + 2 * (i * h + h * o) + 3 * (h + o)),
                "flops": 6 * b * (i * h + h * o)}
    if kind == "dense":
        b, i, o = c["batch"], c["inp"], c["out"]
        # read x, weights, bias, grad_out; write out, gaa, grad_input, grad_weights, grad_bias
        return {"bytes": 4 * (2 * b * i + 3 * b * o + 2 * i * o + 2 * o), "flops": 6 * b * i * o}
    if kind == "attention":
        b, s, d = c["batch"], c["seq"], c["dim"]
        return {"bytes": 4 * 4 * b * s * d, "flops": 4 * b * s * s * d}
    oh, ow = _out_hw(c)
    b, taps = c["batch"], c["c"] * c["ker"] ** 2
    x, y, w = b * c["c"] * c["h"] * c["w"], b * c["oc"] * oh * ow, c["oc"] * taps
    # read x, weights, bias, grad_output; write out, grad_input, grad_weights, grad_bias
    return {"bytes": 4 * (2 * x + 2 * y + 2 * w + 2 * c["oc"]), "flops": 6 * y * taps}


# ------------------------------------------------------------------ inputs
def _rand(gen, *shape):
    """Input activations, as images and sigmoid outputs are: U[0, 1)."""
    return torch.rand(shape, generator=gen, device="cuda", dtype=torch.float32)


def _weight(gen, fan_in, *shape):
    """Dense.init's weights: U[-1, 1) times sqrt(1 / fan_in)."""
    return (_rand(gen, *shape) * 2 - 1) * math.sqrt(1.0 / fan_in)


def _grad(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _empty(*shape):
    return torch.empty(shape, device="cuda", dtype=torch.float32)


def _inputs(case, seed):
    """What a case reads, made from the seed alone."""
    c, kind = case, case["kind"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    if kind in ("gemm", "batched"):
        m, n, k, lay = c["m"], c["n"], c["k"], c["layout"]
        lead = (c["batch"],) if kind == "batched" else ()
        s = {"a": _grad(gen, *lead, *((k, m) if lay == "tn" else (m, k))),
             "b": _weight(gen, k, *lead, *((n, k) if lay == "nt" else (k, n)))}
        if c.get("bias"):
            s["bias"] = _weight(gen, 1, n)
        if c.get("accumulate"):
            s["c0"] = _grad(gen, m, n)
        return s
    if kind == "mlp":
        b, i, h, o = c["batch"], c["inp"], c["hidden"], c["out"]
        return {"x": _rand(gen, b, i), "w1": _weight(gen, i / 2, i, h), "b1": _weight(gen, 1, h),
                "w2": _weight(gen, h, h, o), "b2": _weight(gen, 1, o), "gy": _grad(gen, b, o)}
    if kind == "dense":
        b, i, o = c["batch"], c["inp"], c["out"]
        return {"x": _rand(gen, b, i), "w": _weight(gen, i, i, o), "bias": _weight(gen, 1, o), "gy": _grad(gen, b, o)}
    if kind == "attention":
        shape = (c["batch"], c["seq"], c["dim"])
        return {"q": _grad(gen, *shape), "k": _grad(gen, *shape), "v": _grad(gen, *shape)}
    if kind == "conv":
        oh, ow = _out_hw(c)
        taps = c["c"] * c["ker"] ** 2
        return {"x": _rand(gen, c["batch"], c["c"], c["h"], c["w"]), "w": _weight(gen, taps, c["oc"], taps),
                "bias": _weight(gen, 1, c["oc"]), "gy": _grad(gen, c["batch"], c["oc"], oh, ow)}
    rng = np.random.default_rng(seed)
    m, n, k = c["m"], c["n"], c["k"]
    return {"a": rng.random((m, k), dtype=np.float32),
            "b": ((rng.random((k, n), dtype=np.float32) * 2 - 1) * np.float32(math.sqrt(1.0 / k))).astype(np.float32),
            "bias": rng.random(n, dtype=np.float32)}


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = _inputs(c, seed)
    s["case"] = dict(c)
    if kind == "host":
        s["backend"] = _backend()
        s["out"] = np.empty((c["m"], c["n"]), np.float32)
        return s
    s["ctx"] = _ctx()
    if kind == "gemm":
        s["out"] = _empty(c["m"], c["n"])
    elif kind == "batched":
        s["out"] = _empty(c["batch"], c["m"], c["n"])
    elif kind == "mlp":
        b, i, h, o = c["batch"], c["inp"], c["hidden"], c["out"]
        s.update(h=_empty(b, h), y=_empty(b, o), gaa1=_empty(b, h), gaa2=_empty(b, o), gx=_empty(b, i), gh=_empty(b, h),
                 gw1=_empty(i, h), gw2=_empty(h, o))
        at = (h + 3) // 4 * 4
        s["gb"], s["zeros"] = _empty(at + o).zero_(), torch.zeros(at + o, device="cuda")
        s.update(gb1=s["gb"][:h], gb2=s["gb"][at:])
    elif kind == "dense":
        b, i, o = c["batch"], c["inp"], c["out"]
        s.update(y=_empty(b, o), gaa=_empty(b, o), gx=_empty(b, i), gw=_empty(i, o), gb=_empty(o),
                 zeros=torch.zeros(o, device="cuda"))
    elif kind == "attention":
        s["out"] = _empty(c["batch"], c["seq"], c["dim"])
    else:
        s.update(y=torch.empty_like(s["gy"]), gx=torch.empty_like(s["x"]), gw=torch.empty_like(s["w"]),
                 gb=torch.empty_like(s["bias"]))
    return s


def _p(t):
    return t.data_ptr()


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "host":
        name = "matMulBias" + {"linear": "", "relu": "Relu", "sigmoid": "Sigmoid", "tanh": "Tanh"}[c["act"]]
        getattr(s["backend"], name)(s["a"], s["b"], s["bias"], s["out"], c["m"], c["n"], c["k"])
        return s["out"]
    ctx = s["ctx"]
    if kind in ("gemm", "batched"):
        m, n, k, lay = c["m"], c["n"], c["k"], c["layout"]
        lda, ldb = m if lay == "tn" else k, k if lay == "nt" else n
        if kind == "batched":
            ctx.sgemm_strided_batched(lay, m, n, k, _p(s["a"]), lda, m * k, _p(s["b"]), ldb, k * n, _p(s["out"]), n, m * n,
                                      c["batch"])
            return s["out"]
        if c["accumulate"]:
            # C += A.B onto a running sum: the running sum is set up first, as its producer would
            ctx.copy(_p(s["out"]), _p(s["c0"]), m * n)
        ctx.sgemm(lay, m, n, k, _p(s["a"]), lda, _p(s["b"]), ldb, _p(s["out"]), n, c["accumulate"],
                  _p(s["bias"]) if c["bias"] else None, c["act"])
        return s["out"]
    if kind == "mlp":
        b, i, h, o = c["batch"], c["inp"], c["hidden"], c["out"]
        # the bias gradients accumulate: a training loop clears them before each step (here one buffer holds both)
        ctx.copy(_p(s["gb"]), _p(s["zeros"]), s["gb"].numel())
        ctx.dense_pair_forward(c["act"], _p(s["x"]), _p(s["w1"]), _p(s["b1"]), _p(s["h"]), "linear", _p(s["w2"]), _p(s["b2"]),
                               _p(s["y"]), b, i, h, o)
        ctx.dense_pair_backward(c["act"], _p(s["x"]), _p(s["w1"]), _p(s["h"]), _p(s["gaa1"]), _p(s["gx"]), _p(s["gw1"]),
                                _p(s["gb1"]), "linear", _p(s["w2"]), _p(s["y"]), _p(s["gy"]), _p(s["gaa2"]), _p(s["gh"]),
                                _p(s["gw2"]), _p(s["gb2"]), b, i, h, o)
        return {k: s[k] for k in ("h", "y", "gaa1", "gaa2", "gx", "gh", "gw1", "gw2", "gb1", "gb2")}
    if kind == "dense":
        b, i, o = c["batch"], c["inp"], c["out"]
        ctx.copy(_p(s["gb"]), _p(s["zeros"]), o)  # the bias gradient accumulates: cleared before each step
        ctx.sgemm("nn", b, o, i, _p(s["x"]), i, _p(s["w"]), o, _p(s["y"]), o, False, _p(s["bias"]), c["act"])
        ctx.dense_backward(c["act"], _p(s["x"]), _p(s["w"]), _p(s["y"]), _p(s["gy"]), _p(s["gaa"]), _p(s["gx"]), _p(s["gw"]),
                           _p(s["gb"]), b, i, o)
        return {k: s[k] for k in ("y", "gaa", "gx", "gw", "gb")}
    if kind == "attention":
        ctx.attention_forward(_p(s["q"]), _p(s["k"]), _p(s["v"]), _p(s["out"]), c["batch"], c["seq"], c["dim"],
                              1.0 / math.sqrt(c["dim"]))
        return s["out"]
    oh, ow = _out_hw(c)
    geom = (c["batch"], c["c"], c["oc"], c["ker"], c["ker"], c["h"], c["w"], oh, ow, c["stride"], c["stride"], c["pad"],
            c["pad"])
    forward, backward = ((ctx.conv2d_forward_im2col, ctx.conv2d_backward_im2col) if c["order"] == "im2col" else
                         (ctx.conv2d_forward_direct, ctx.conv2d_backward_direct))
    forward(_p(s["x"]), _p(s["w"]), _p(s["bias"]), _p(s["y"]), *geom)
    backward(_p(s["x"]), _p(s["w"]), _p(s["gy"]), _p(s["gx"]), _p(s["gw"]), _p(s["gb"]), *geom)
    return {k: s[k] for k in ("y", "gx", "gw", "gb")}


# ------------------------------------------------------------------ what the results have to be
#: Largest relative error (2-norm) another float32 implementation shows: about four times what the paths show against
#: 64 bits (1.6e-6 for sums of 8192 terms, 6e-7 to 8e-7 for a Dense step, attention and a convolution's gradients).
_REL = {"gemm": 6e-6, "batched": 2e-6, "mlp": 4e-6, "dense": 4e-6, "attention": 4e-6, "conv": 4e-6, "host": 2e-6}


def tolerance(case):
    return {"rel": _REL[case["kind"]]}


def _act64(name, v):
    return {"linear": lambda t: t, "relu": lambda t: t.clamp(min=0), "sigmoid": torch.sigmoid, "tanh": torch.tanh}[name](v)


def _dact64(name, y, g):
    if name == "linear":
        return g
    if name == "relu":
        return torch.where(y > 0, g, torch.zeros_like(g))
    return g * (y * (1 - y) if name == "sigmoid" else 1 - y * y)


def _col64(c, x):
    """[batch * OH * OW][taps] in the case's weight order."""
    f = torch.nn.functional.unfold(x, c["ker"], padding=c["pad"], stride=c["stride"])  # [b][C * k * k][OH * OW]
    b, _, p = f.shape
    f = f.reshape(b, c["c"], c["ker"] ** 2, p)
    f = f.permute(0, 3, 2, 1) if c["order"] == "im2col" else f.permute(0, 3, 1, 2)
    return f.reshape(b * p, -1).contiguous()


def _im64(c, col):
    """The adjoint of _col64."""
    oh, ow = _out_hw(c)
    b, kk = c["batch"], c["ker"] ** 2
    if c["order"] == "im2col":
        f = col.reshape(b, oh * ow, kk, c["c"]).permute(0, 3, 2, 1)
    else:
        f = col.reshape(b, oh * ow, c["c"], kk).permute(0, 2, 3, 1)
    f = f.reshape(b, c["c"] * kk, oh * ow).contiguous()
    return torch.nn.functional.fold(f, (c["h"], c["w"]), c["ker"], padding=c["pad"], stride=c["stride"])


def exact(case, seed):
    c, kind = case, case["kind"]
    s = _inputs(c, seed)
    if kind == "host":
        v = s["a"].astype(np.float64) @ s["b"].astype(np.float64) + s["bias"].astype(np.float64)
        return _act64(c["act"], torch.from_numpy(v)).numpy()
    s = {k: t.double() for k, t in s.items()}
    if kind in ("gemm", "batched"):
        a = s["a"].transpose(-1, -2).contiguous() if c["layout"] == "tn" else s["a"]
        b = s["b"].transpose(-1, -2).contiguous() if c["layout"] == "nt" else s["b"]
        v = torch.matmul(a, b)
        if "c0" in s:
            v += s["c0"]
        if "bias" in s:
            v += s["bias"]
        return _act64(c.get("act", "linear"), v)
    if kind == "mlp":
        h = _act64(c["act"], s["x"] @ s["w1"] + s["b1"])
        y = h @ s["w2"] + s["b2"]
        gaa2 = s["gy"]
        gh = gaa2 @ s["w2"].t().contiguous()
        gaa1 = _dact64(c["act"], h, gh)
        return {"h": h, "y": y, "gaa1": gaa1, "gaa2": gaa2, "gx": gaa1 @ s["w1"].t().contiguous(), "gh": gh,
                "gw1": s["x"].t().contiguous() @ gaa1, "gw2": h.t().contiguous() @ gaa2, "gb1": gaa1.sum(0), "gb2": gaa2.sum(0)}
    if kind == "dense":
        y = _act64(c["act"], s["x"] @ s["w"] + s["bias"])
        gaa = _dact64(c["act"], y, s["gy"])
        return {"y": y, "gaa": gaa, "gx": gaa @ s["w"].t().contiguous(), "gw": s["x"].t().contiguous() @ gaa, "gb": gaa.sum(0)}
    if kind == "attention":
        out = []
        for q, k, v in zip(s["q"], s["k"], s["v"]):  # one head at a time: the scores of all of them would not fit
            out.append(torch.softmax(q @ k.t().contiguous() / math.sqrt(c["dim"]), -1) @ v)
        return torch.stack(out)
    oh, ow = _out_hw(c)
    b, oc = c["batch"], c["oc"]
    col = _col64(c, s["x"])
    y = (col @ s["w"].t().contiguous() + s["bias"]).reshape(b, oh * ow, oc).permute(0, 2, 1).reshape(b, oc, oh, ow).contiguous()
    # the im2col branch reads grad_output's memory as [batch * OH * OW][OC] for both gradients (the reference's contract)
    if c["order"] == "im2col":
        g = s["gy"].reshape(b * oh * ow, oc)
    else:
        g = s["gy"].reshape(b, oc, oh * ow).permute(0, 2, 1).reshape(b * oh * ow, oc).contiguous()
    return {"y": y, "gx": _im64(c, g @ s["w"]), "gw": g.t().contiguous() @ col, "gb": s["gy"].sum((0, 2, 3))}
