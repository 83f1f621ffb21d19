"""The work that programs on this library have it do, as measurable cases.

A program on this library either calls the op layer itself (``forward_op`` / ``backward_op``, the
tensorutils reductions, the fused row and bias patterns, ``Adam``) on device tensors, or builds a
``Graph`` and trains it through ``Model`` and ``Adam``. Each kind of case below is one of these
uses over the sizes it meets; every call is queued (``init(asynchronous=True)``), as a program
that trains for many steps does. Data is fp32, the library's one type.

Inputs are drawn with torch from the seed alone and copied into the library's tensors; results
are the library's own buffers, seen as torch tensors. Gradients accumulate from pass to pass, as
over micro-batches, except in the training steps, which clear them.
"""
import math
import random

import numpy as np
import torch

import mantle_amd as m

OP = m.OP
BINARY = (OP.ADD, OP.SUB, OP.MUL, OP.DIV)
UNARY = (OP.EXP, OP.LOG, OP.SIGMOID, OP.RELU, OP.TANH)
SLOPE, CLIP_LO, CLIP_HI = 0.1, -1.1, 1.1
LR, B1, B2, EPS = 1e-3, 0.9, 0.999, 1e-8
MAX_ELEMENTS = 1 << 27


# ---------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------
def listed():
    return [
        # one training step of a deep model of small layers (24 of MUL(w) -> ADD(b) -> RELU over
        # [32, 32]): zero_grad, forward, backward, Adam; latency and launch count
        {"name": "step_deep_small", "kind": "step", "layers": 24, "rows": 32, "width": 32, "act": "RELU",
         "fuse": False},
        # the classifier head over [2^20, 10] in the executor's default form: MAX, SUB, EXP, SUM,
        # DIV, LOG, MUL(target), MEAN and their backward, one kernel per node
        {"name": "head_1m_x_10", "kind": "head", "rows": 1 << 20, "classes": 10, "fuse": False},
        # a convolution's bias and activation, forward and backward: x [256, 32, 28, 28] + [1, 32, 1, 1]
        {"name": "bias_relu_nchw", "kind": "bias", "n": 256, "c": 32, "s": 784, "fuse": True},
        # a Linear layer's bias and activation over a batch: x [16384, 1000] + [1, 1000]
        {"name": "bias_relu_linear", "kind": "bias", "n": 16384, "c": 1000, "s": 1, "fuse": True},
        # every elementwise op, forward and backward, on a tensor as small as a layer's bias
        {"name": "elementwise_small", "kind": "ew", "ops": "all", "n": 1023, "scalar": False},
        # the binary ops, forward and both gradients, on tensors far larger than any cache
        {"name": "binary_large", "kind": "ew", "ops": "binary", "n": 1 << 27, "scalar": False},
        # SUB, MUL, DIV of feature maps by a per-channel tensor, with both gradients: a 27 x 27 map
        # has an odd number of pixels, as most of the late maps of a convolutional network do
        {"name": "channel_27x27", "kind": "bcast", "a": 256, "b": 96, "c": 729, "pattern": "chan"},
        # SUM, MEAN, MAX over a batch axis, forward and backward
        {"name": "reduce_axis0_8192", "kind": "reduce", "a": 1, "b": 8192, "c": 8192, "whole": False},
        # the same over the middle axis of a tensor with no even size
        {"name": "reduce_middle_odd", "kind": "reduce", "a": 33, "b": 1025, "c": 1023, "whole": False},
        # CrossEntropyLoss over 1000 classes, forward and backward
        {"name": "cross_entropy_1000", "kind": "rows", "graph": "ce", "rows": 32768, "classes": 1000},
        # normalising rows with the reductions: (x - mean) / std over the last axis
        {"name": "normalise_rows", "kind": "norm", "a": 32768, "b": 1023, "c": 1},
        # an optimizer step over a model of 400 parameters of 1 to 2^18 elements
        {"name": "adam_400_tensors", "kind": "adam", "tensors": 400, "largest": 1 << 18},
    ]


def _size(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "head", "bias", "ew", "bcast", "reduce", "rows", "norm", "adam"])
    if kind == "step":
        rows, width = _size(rng, 1, 16384), _size(rng, 4, 2048)
        return {"kind": kind, "layers": _size(rng, 1, min(24, max(1, (1 << 25) // (rows * width)))), "rows": rows,
                "width": width, "act": rng.choice(["RELU", "SIGMOID", "TANH"]), "fuse": rng.random() < 0.5}
    if kind == "head":
        classes = _size(rng, 2, 2047)
        return {"kind": kind, "rows": _size(rng, 16, (1 << 24) // classes), "classes": classes,
                "fuse": rng.random() < 0.5}
    if kind == "bias":
        if rng.random() < 0.5:  # a Linear layer's [rows, features]
            c = _size(rng, 8, 4096)
            return {"kind": kind, "n": _size(rng, 16, (1 << 24) // c), "c": c, "s": 1, "fuse": rng.random() < 0.5}
        s = _size(rng, 4, 128) ** 2  # a convolution's [images, channels, side, side]
        c = _size(rng, 3, 512)
        return {"kind": kind, "n": _size(rng, 1, max(1, (1 << 24) // (c * s))), "c": c, "s": s,
                "fuse": rng.random() < 0.5}
    if kind == "ew":
        ops = rng.choice(["binary", "unary", "pow", "adjacent", "all"])
        return {"kind": kind, "ops": ops, "n": _size(rng, 32, 1 << (22 if ops == "all" else 26)),
                "scalar": rng.random() < 0.25}
    if kind == "bcast":
        c, b = _size(rng, 4, 4096), _size(rng, 2, 512)
        return {"kind": kind, "a": _size(rng, 2, max(2, (1 << 24) // (b * c))), "b": b, "c": c,
                "pattern": rng.choice(["chan", "row", "col", "mid", "outer"])}
    if kind == "reduce":
        axis = rng.choice([0, 1, 2, None])
        if axis is None:
            return {"kind": kind, "a": 1, "b": _size(rng, 1 << 10, 1 << 26), "c": 1, "whole": True}
        b = _size(rng, 2, 1 << 14)
        c = 1 if axis == 2 else _size(rng, 2, 1 << 13)
        a = 1 if axis == 0 else _size(rng, 2, max(2, (1 << 26) // (b * c)))
        return {"kind": kind, "a": a, "b": b, "c": c, "whole": False}
    if kind == "rows":
        classes = _size(rng, 2, 2047)
        return {"kind": kind, "graph": rng.choice(["ce", "head", "softmax", "logsoftmax"]),
                "rows": _size(rng, 16, (1 << 25) // classes), "classes": classes}
    if kind == "norm":
        b = _size(rng, 16, 1 << 14)
        c = rng.choice([1, _size(rng, 2, 1 << 11)])
        return {"kind": kind, "a": _size(rng, 1, max(1, (1 << 25) // (b * c))), "b": b, "c": c}
    return {"kind": "adam", "tensors": _size(rng, 1, 1000), "largest": _size(rng, 64, 1 << 17)}


def _adam_sizes(case):
    r = random.Random(case["tensors"])
    return [r.randint(1, case["largest"]) for _ in range(case["tensors"])]


def _bcast_shapes(case):
    a, b, c = case["a"], case["b"], case["c"]
    full = (a, b, c)
    return {"chan": (full, (1, b, 1)), "row": (full, (a, b, 1)), "col": (full, (1, 1, c)), "mid": (full, (a, 1, c)),
            "outer": ((a, 1, c), (1, b, 1))}[case["pattern"]]


def _ew_ops(case):
    ops = case["ops"]
    return {"binary": BINARY, "unary": UNARY, "pow": (OP.POW,), "adjacent": (OP.FMA, OP.LEAKYRELU, OP.CLIP),
            "all": BINARY + UNARY + (OP.POW, OP.FMA, OP.LEAKYRELU, OP.CLIP)}[ops]


def _bias_shapes(case):
    n, c, s = case["n"], case["c"], case["s"]
    if s == 1:
        return (n, c), (1, c)
    side = math.isqrt(s)
    return (n, c, side, s // side), (1, c, 1, 1)


# ---------------------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------------------
class _Draw:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, shape, mean=0.0, std=1.0):
        return torch.empty(shape, device="cuda").normal_(mean, std, generator=self.g)

    def uniform(self, shape, lo, hi):
        return torch.empty(shape, device="cuda").uniform_(lo, hi, generator=self.g)

    def onehot(self, rows, classes):
        k = torch.randint(0, classes, (rows, 1), device="cuda", generator=self.g)
        return torch.zeros((rows, classes), device="cuda").scatter_(1, k, 1.0)


def _inputs(case, seed):
    """{name: torch tensor}, and for a step its layers' weights and biases."""
    d, kind = _Draw(seed), case["kind"]
    if kind == "step":
        t = {"x": d.normal((case["rows"], case["width"]))}
        for i in range(case["layers"]):
            t["w%d" % i] = d.normal((1, case["width"]), 1.0, 0.1)
            t["b%d" % i] = d.normal((1, case["width"]), 0.0, 0.1)
        return t
    if kind in ("head", "rows"):
        r, k = case["rows"], case["classes"]
        t = {"x": d.normal((r, k), 0.0, 2.0)}
        if kind == "head" or case["graph"] in ("ce", "head"):
            t["t"] = d.onehot(r, k)
            if kind == "rows":
                t["ug"] = torch.ones(1, device="cuda")
        else:
            t["ug"] = d.normal((r, k))
        return t
    if kind == "bias":
        sx, sb = _bias_shapes(case)
        return {"x": d.normal(sx), "bias": d.normal(sb, 0.0, 0.1), "ug": d.normal(sx)}
    if kind == "ew":
        n = case["n"]
        t = {"ug": d.normal((n,))}
        ops = _ew_ops(case)
        if OP.ADD in ops:
            t["a"] = d.uniform((n,), -1.0, 1.0)
            t["b"] = d.uniform((1 if case["scalar"] else n,), 0.5, 2.0)
        if OP.EXP in ops or OP.LEAKYRELU in ops:
            t["x"] = d.normal((n,), 0.0, 3.0)
        if OP.LOG in ops or OP.POW in ops:
            t["p"] = d.uniform((n,), 0.1, 4.0)
        if OP.POW in ops:
            t["e"] = d.uniform((1,), 0.5, 3.0)
        if OP.FMA in ops:
            t["y"], t["z"] = d.normal((n,)), d.normal((n,))
        return t
    if kind == "bcast":
        s1, s2 = _bcast_shapes(case)
        return {"t1": d.normal(s1), "t2": d.uniform(s2, 0.5, 2.0), "ug": d.normal((case["a"], case["b"], case["c"]))}
    if kind == "reduce":
        if case["whole"]:
            return {"x": d.normal((case["b"],)), "ug": d.normal((1,))}
        return {"x": d.normal((case["a"], case["b"], case["c"])), "ug": d.normal((case["a"], 1, case["c"]))}
    if kind == "norm":
        return {"x": d.normal((case["a"], case["b"], case["c"]), 0.5, 2.0)}
    t = {}
    for i, n in enumerate(_adam_sizes(case)):
        t["p%d" % i] = d.normal((n,))
        t["g%d" % i] = d.normal((n,), 0.0, 0.1)
    return t


# ---------------------------------------------------------------------------------------
# the library's tensors
# ---------------------------------------------------------------------------------------
class _Span:
    """A library tensor's memory, for torch."""

    def __init__(self, t):
        self.owner = t
        self.__cuda_array_interface__ = {"shape": t.shape().dims, "typestr": "<f4", "data": (t.ptr, False),
                                         "strides": None, "version": 2}


def _view(t):
    return torch.as_tensor(_Span(t), device="cuda")


class _State:
    """Library tensors by name (.t) with their torch views (.v), and what a program keeps beside."""

    def __init__(self, case):
        m.init(0, asynchronous=True)
        self.case, self.t, self.v = case, {}, {}

    def new(self, name, shape):
        self.t[name] = m.Tensor(tuple(shape))
        self.v[name] = _view(self.t[name])
        return self.t[name]

    def load(self, values):
        """Inputs into tensors of their own; returns when they are there."""
        for k, v in values.items():
            if k not in self.t:
                self.new(k, v.shape)
        m.sync()  # the new tensors' zeroes
        for k, v in values.items():
            self.v[k].copy_(v)
        torch.cuda.synchronize()


def _numpy(t):
    return t.cpu().numpy()


def _prepare_step(s, values):
    g = m.Graph()
    x = g.input(tuple(values["x"].shape))
    h, params = x, []
    for i in range(s.case["layers"]):
        w = g.param(tuple(values["w%d" % i].shape), init=_numpy(values["w%d" % i]))
        b = g.param(tuple(values["b%d" % i].shape), init=_numpy(values["b%d" % i]))
        h = g.op(getattr(OP, s.case["act"]), g.op(OP.ADD, g.op(OP.MUL, h, w), b))
        params += [w, b]
    g.loss(g.op(OP.MEAN, h))
    s.model = m.Model(g, fuse_bias_relu=s.case["fuse"])
    s.opt = m.Adam(s.model.parameters, lr=LR, beta1=B1, beta2=B2, epsilon=EPS)
    s.load({"x": values["x"]})
    # the arena's own spans: every parameter and every gradient of the model, slot by slot
    s.out = {"loss": _view(s.model.parameters.tensors[g.loss_out])}
    s.flat = [_view(s.model.parameters.tensors[p]) for p in params], [_view(s.model.parameters.grads[p]) for p in params]


def _prepare_head(s, values):
    rows, k = s.case["rows"], s.case["classes"]
    g = m.Graph()
    x, t = g.input((rows, k), trainable=True), g.input((rows, k))
    e = g.op(OP.EXP, g.op(OP.SUB, x, g.op(OP.MAX, x, attributes={"axis": 1})))
    sm = g.op(OP.DIV, e, g.op(OP.SUM, e, attributes={"axis": 1}))
    g.loss(g.op(OP.MEAN, g.op(OP.MUL, g.op(OP.LOG, sm), t)))
    s.model = m.Model(g, fuse_rows=s.case["fuse"])
    s.load(values)
    s.out = {"loss": _view(s.model.parameters.tensors[g.loss_out]), "grad_x": _view(s.model.parameters.grads[x])}


def prepare(case, seed):
    s, values = _State(case), _inputs(case, seed)
    kind = case["kind"]
    if kind == "step":
        _prepare_step(s, values)
        return s
    if kind == "head":
        _prepare_head(s, values)
        return s
    if kind == "bias":
        sx, sb = _bias_shapes(case)
        for k in ("y", "r", "gy", "gx"):
            s.new(k, sx)
        s.new("gb", sb)
    elif kind == "ew":
        n = case["n"]
        for op in _ew_ops(case):
            s.new("f%d" % op, (n,))
            s.new("g%d" % op, (n,))
            if op in BINARY:
                s.new("h%d" % op, values["b"].shape)
            if op == OP.POW:
                s.new("h%d" % op, (1,))
            if op == OP.FMA:
                s.new("h%d" % op, (n,))
                s.new("i%d" % op, (n,))
    elif kind == "bcast":
        for op in (OP.SUB, OP.MUL, OP.DIV):
            s.new("f%d" % op, values["ug"].shape)
            s.new("g%d" % op, values["t1"].shape)
            s.new("h%d" % op, values["t2"].shape)
    elif kind == "reduce":
        for op in (OP.SUM, OP.MEAN, OP.MAX):
            s.new("f%d" % op, values["ug"].shape)
            s.new("g%d" % op, values["x"].shape)
    elif kind == "rows":
        s.new("out", (1,) if case["graph"] in ("ce", "head") else values["x"].shape)
        s.new("gx", values["x"].shape)
    elif kind == "norm":
        line = (case["a"], 1, case["c"])
        for k, shape in (("mean", line), ("std", line), ("centred", values["x"].shape), ("y", values["x"].shape)):
            s.new(k, shape)
    s.load(values)
    if kind == "adam":
        n = case["tensors"]
        s.opt = m.Adam([(s.t["p%d" % i], s.t["g%d" % i]) for i in range(n)], lr=LR, beta1=B1, beta2=B2, epsilon=EPS)
        s.first = [_view(t) for t in s.opt.momentum_grads]
        s.second = [_view(t) for t in s.opt.rms_grads]
        m.sync()
    return s


# ---------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------
def _join(tensors):
    """Tensors of many sizes as one result: up to 16 of them as they are, or the smallest, the
    largest and 14 between (a result holds few arrays)."""
    if len(tensors) <= 16:
        return list(tensors)
    order = sorted(range(len(tensors)), key=lambda i: (tensors[i].numel(), i))
    return [tensors[order[(len(order) - 1) * k // 15]] for k in range(16)]


def _run_ew(s):
    t, case = s.t, s.case
    for op in _ew_ops(case):
        f, g = t["f%d" % op], t["g%d" % op]
        if op in BINARY:
            m.forward_op(op, f, t["a"], t["b"])
            m.backward_op_both(op, t["ug"], t["a"], t["b"], g, t["h%d" % op])
        elif op == OP.POW:
            m.forward_op(op, f, t["p"], t["e"])
            m.backward_op_both(op, t["ug"], t["p"], t["e"], g, t["h%d" % op])
        elif op == OP.FMA:
            m.forward_op(op, f, t["x"], t["y"], t3=t["z"])
            for i, k in enumerate("ghi"):
                m.backward_op(i, op, t["ug"], t["x"], t["y"], t["%s%d" % (k, op)], t3=t["z"])
        else:
            at = {OP.LEAKYRELU: {"negative_slope": SLOPE}, OP.CLIP: {"min": CLIP_LO, "max": CLIP_HI}}.get(op)
            x = t["p"] if op == OP.LOG else t["x"]
            m.forward_op(op, f, x, attributes=at)
            m.backward_op(0, op, t["ug"], x, None, g, attributes=at)
    return {k: v for k, v in s.v.items() if k[0] in "fghi"}


def run(s):
    case, t, v = s.case, s.t, s.v
    kind = case["kind"]
    if kind == "step":
        s.opt.zero_grad()
        s.model.forward(t["x"])
        s.model.backward()
        s.opt.step()
        return dict(s.out, params=_join(s.flat[0]), grads=_join(s.flat[1]))
    if kind == "head":
        s.model.parameters.grads.set_zero()
        s.model.forward(t["x"], t["t"])
        s.model.backward()
        return s.out
    if kind == "bias":
        if case["fuse"]:
            m.bias_relu_forward(t["y"], t["r"], t["x"], t["bias"])
            m.bias_relu_backward(t["ug"], t["y"], t["bias"].shape(), t["gx"], t["gb"], t["gy"])
        else:
            m.forward_op(OP.ADD, t["y"], t["x"], t["bias"])
            m.forward_op(OP.RELU, t["r"], t["y"])
            m.backward_op(0, OP.RELU, t["ug"], t["y"], None, t["gy"])
            m.backward_op(0, OP.ADD, t["gy"], t["x"], t["bias"], t["gx"])
            m.backward_op(1, OP.ADD, t["gy"], t["x"], t["bias"], t["gb"])
        return {k: v[k] for k in ("y", "r", "gy", "gx", "gb")}
    if kind == "ew":
        return _run_ew(s)
    if kind == "bcast":
        for op in (OP.SUB, OP.MUL, OP.DIV):
            m.forward_op(op, t["f%d" % op], t["t1"], t["t2"])
            m.backward_op(0, op, t["ug"], t["t1"], t["t2"], t["g%d" % op])
            m.backward_op(1, op, t["ug"], t["t1"], t["t2"], t["h%d" % op])
        return {k: x for k, x in v.items() if k[0] in "fgh"}
    if kind == "reduce":
        at = None if case["whole"] else {"axis": 1}
        for op in (OP.SUM, OP.MEAN, OP.MAX):
            m.forward_op(op, t["f%d" % op], t["x"], attributes=at)
            m.backward_op(0, op, t["ug"], t["x"], None, t["g%d" % op], attributes=at)
        return {k: x for k, x in v.items() if k[0] in "fg"}
    if kind == "rows":
        graph = case["graph"]
        if graph == "ce":
            m.cross_entropy_forward(t["out"], t["x"], t["t"])
            m.cross_entropy_backward(t["gx"], t["x"], t["t"], t["ug"])
        elif graph == "head":
            m.softmax_log_mul_mean_forward(t["out"], t["x"], t["t"])
            m.softmax_log_mul_mean_backward(t["gx"], t["x"], t["t"], t["ug"])
        elif graph == "softmax":
            m.softmax_forward(t["out"], t["x"])
            m.softmax_backward(t["gx"], t["x"], t["ug"])
        else:
            m.logsoftmax_forward(t["out"], t["x"])
            m.logsoftmax_backward(t["gx"], t["x"], t["ug"])
        return {"out": v["out"], "gx": v["gx"]}
    if kind == "norm":
        m.tmean(t["x"], 1, t["mean"])
        m.tstd(t["x"], 1, t["std"])
        m.forward_op(OP.SUB, t["centred"], t["x"], t["mean"])
        m.forward_op(OP.DIV, t["y"], t["centred"], t["std"])
        return {k: v[k] for k in ("mean", "std", "y")}
    s.opt.step()
    n = case["tensors"]
    return {"p": _join([v["p%d" % i] for i in range(n)]), "m": _join(s.first), "v": _join(s.second)}


# ---------------------------------------------------------------------------------------
# the least that a pass moves and computes
# ---------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "step":  # x read; loss, every parameter, gradient and both moments once over
        n, p = case["rows"] * case["width"], 2 * case["layers"] * case["width"]
        return {"bytes": 4 * (n + 8 * p + 1), "flops": 12 * n * case["layers"] + 14 * p}
    if kind == "head":
        n = case["rows"] * case["classes"]
        return {"bytes": 12 * n, "flops": 40 * n}
    if kind == "bias":  # x, ug read; y, r written; both gradients read and written; the bias and its gradient
        n = case["n"] * case["c"] * case["s"]
        return {"bytes": 32 * n + 12 * case["c"], "flops": 5 * n}
    if kind == "ew":
        n, b, f = case["n"], 0, 0
        for op in _ew_ops(case):
            if op in BINARY:  # forward; ug (and for MUL, DIV the operands) read, both gradients read and written
                if case["scalar"]:
                    b += 8 + 12 + (4 if op in (OP.MUL, OP.DIV) else 0)
                else:
                    b += 12 + 20 + (8 if op in (OP.MUL, OP.DIV) else 0)
                f += 6
            elif op == OP.POW:
                b += 8 + 16
                f += 60
            elif op == OP.FMA:
                b += 16 + 4 + 8 + 24
                f += 7
            else:
                b += 8 + 16
                f += 40
        return {"bytes": b * n, "flops": f * n}
    if kind == "bcast":
        s1, s2 = _bcast_shapes(case)
        n, n1, n2 = case["a"] * case["b"] * case["c"], math.prod(s1), math.prod(s2)
        # forward reads both and writes n; the gradients read ug (and for MUL, DIV both operands)
        return {"bytes": 4 * (3 * (n1 + n2 + n) + 3 * (n + 2 * n1 + 2 * n2) + 2 * (n1 + n2)), "flops": 18 * n}
    if kind == "reduce":  # three forwards read x; three gradients read and written, MAX reading x again
        n, o = case["a"] * case["b"] * case["c"], case["a"] * case["c"]
        return {"bytes": 4 * (3 * n + 3 * o + 6 * n + n + 3 * o), "flops": 10 * n}
    if kind == "rows":
        n = case["rows"] * case["classes"]
        return {"bytes": 24 * n, "flops": 50 * n}
    if kind == "norm":  # x read, y and the centred values written
        n, o = case["a"] * case["b"] * case["c"], case["a"] * case["c"]
        return {"bytes": 4 * (3 * n + 2 * o), "flops": 8 * n}
    n = sum(_adam_sizes(case))
    return {"bytes": 28 * n, "flops": 14 * n}


def tolerance(case):
    """Against 64 bits the library's results are off by up to 3e-7 (Adam's moments, whose factors
    1 - beta are rounded to 32 bits; sums in tree order) and by 1e-7 elsewhere. Kinds whose
    results hold sums of signed terms, which nearly cancel at some of the drawn sizes, take what
    another order of a 32-bit sum gives there."""
    return {"rel": 1e-6 if case["kind"] in ("adam", "rows", "head", "norm") else 1e-5}


# ---------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------
def _adam64(p, g):
    """Adam's first step from zero moments: (p, m, v)."""
    mm, vv = (1 - B1) * g, (1 - B2) * g * g
    return p - LR * ((mm / (1 - B1)) / (torch.sqrt(vv / (1 - B2)) + EPS)), mm, vv


def _unary64(op, x, ug):
    if op == OP.EXP:
        e = x.exp()
        return e, e * ug
    if op == OP.LOG:
        return x.log(), ug / x
    if op == OP.SIGMOID:
        y = torch.sigmoid(x)
        return y, y * (1 - y) * ug
    if op == OP.RELU:
        return x.clamp(min=0), (x > 0) * ug
    if op == OP.TANH:
        y = torch.tanh(x)
        return y, (1 - y * y) * ug
    if op == OP.LEAKYRELU:
        k = np.float64(np.float32(SLOPE))
        return torch.where(x > 0, x, x * k), torch.where(x > 0, ug, ug * k)
    lo, hi = np.float64(np.float32(CLIP_LO)), np.float64(np.float32(CLIP_HI))
    return x.clamp(lo, hi), torch.where((x >= lo) & (x <= hi), ug, torch.zeros_like(ug))


def _binary64(op, a, b, ug):
    """(result, gradient of a, gradient of b), the gradients of broadcast operands summed."""
    if op == OP.ADD:
        r, ga, gb = a + b, ug, ug
    elif op == OP.SUB:
        r, ga, gb = a - b, ug, -ug
    elif op == OP.MUL:
        r, ga, gb = a * b, ug * b, ug * a
    else:
        r, ga, gb = a / b, ug / b, -a / (b * b) * ug
    return r, ga.sum_to_size(a.shape), gb.sum_to_size(b.shape)


def exact(case, seed):
    kind = case["kind"]
    t = {k: v.double() for k, v in _inputs(case, seed).items()}
    if kind == "step":
        n = case["layers"]
        names = [c + str(i) for i in range(n) for c in "wb"]
        p = [t[k].requires_grad_(True) for k in names]
        act = {"RELU": torch.relu, "SIGMOID": torch.sigmoid, "TANH": torch.tanh}[case["act"]]
        h = t["x"]
        for i in range(n):
            h = act(h * t["w%d" % i] + t["b%d" % i])
        loss = h.mean().reshape(1)
        loss.backward()
        return {"loss": loss.detach(), "params": _join([_adam64(x.detach(), x.grad)[0] for x in p]),
                "grads": _join([x.grad for x in p])}
    if kind in ("head", "rows"):
        x = t["x"].requires_grad_(True)
        graph = "head" if kind == "head" else case["graph"]
        if graph == "head":
            out = (torch.softmax(x, 1).log() * t["t"]).mean().reshape(1)
        elif graph == "ce":
            out = (-(torch.log_softmax(x, 1) * t["t"]).sum() / case["rows"]).reshape(1)
        else:
            out = torch.softmax(x, 1) if graph == "softmax" else torch.log_softmax(x, 1)
        out.backward(torch.ones(1, dtype=torch.float64, device="cuda") if kind == "head" else t["ug"])
        return {"loss" if kind == "head" else "out": out.detach(), "grad_x" if kind == "head" else "gx": x.grad}
    if kind == "bias":
        y = t["x"] + t["bias"]
        gy = (y > 0) * t["ug"]
        return {"y": y, "r": y.clamp(min=0), "gy": gy, "gx": gy, "gb": gy.sum_to_size(t["bias"].shape)}
    if kind == "ew":
        out = {}
        for op in _ew_ops(case):
            if op in BINARY:
                out["f%d" % op], out["g%d" % op], out["h%d" % op] = _binary64(op, t["a"], t["b"], t["ug"])
            elif op == OP.POW:  # the forward takes the exponent's whole part, the gradients the exponent
                p, e = t["p"], float(t["e"][0])
                out["f%d" % op] = p ** int(e)
                out["g%d" % op] = e * p ** (e - 1) * t["ug"]
                out["h%d" % op] = (p ** e * p.log() * t["ug"]).sum().reshape(1)
            elif op == OP.FMA:
                out["f%d" % op] = t["x"] * t["y"] + t["z"]
                out["g%d" % op], out["h%d" % op], out["i%d" % op] = t["ug"] * t["y"], t["ug"] * t["x"], t["ug"]
            else:
                out["f%d" % op], out["g%d" % op] = _unary64(op, t["p"] if op == OP.LOG else t["x"], t["ug"])
        return out
    if kind == "bcast":
        out = {}
        for op in (OP.SUB, OP.MUL, OP.DIV):
            out["f%d" % op], out["g%d" % op], out["h%d" % op] = _binary64(op, t["t1"], t["t2"], t["ug"])
        return out
    if kind == "reduce":
        x, ug = t["x"], t["ug"]
        ax = 0 if case["whole"] else 1
        top = x.amax(ax, keepdim=True)
        hit = x == top
        return {"f%d" % OP.SUM: x.sum(ax, keepdim=True), "f%d" % OP.MEAN: x.mean(ax, keepdim=True), "f%d" % OP.MAX: top,
                "g%d" % OP.SUM: ug.expand_as(x), "g%d" % OP.MEAN: (ug / case["b"]).expand_as(x),
                "g%d" % OP.MAX: hit * (ug / hit.sum(ax, keepdim=True))}
    if kind == "norm":
        x = t["x"]
        mean, std = x.mean(1, keepdim=True), x.std(1, keepdim=True, correction=0)
        return {"mean": mean, "std": std, "y": (x - mean) / std}
    got = [_adam64(t["p%d" % i], t["g%d" % i]) for i in range(case["tensors"])]
    return {"p": _join([g[0] for g in got]), "m": _join([g[1] for g in got]), "v": _join([g[2] for g in got])}
