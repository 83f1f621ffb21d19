"""The executor's programs (runs of nodes as one launch) at the edges of their forms: one slab of
short and long column sums, several slabs with a short last one, widths that are and are not a
multiple of 4, rows by thread and by wavefront, and views just past a limit. Every tensor and
gradient slot against the oracle running the graph node by node."""
import numpy as np
import pytest

from mantle_amd import synth
from util import O, OPS, GpuEngine, Graph, OracleEngine, assert_bitexact, assert_sum_close, native_graph

pytestmark = pytest.mark.gpu
ORC = OracleEngine()


@pytest.fixture(scope="module")
def gpu():
    return GpuEngine()


@pytest.fixture(autouse=True)
def _nelts():
    O.set_nelts(32)
    yield


# one slab (64 and 65 rows: the column sums' orders), its limit of 8192 elements, several slabs
# (a last one of few rows), the widths 4096 / 8 rows and past it
SHAPES = [(1, 7), (2, 2), (5, 64), (64, 33), (65, 33), (64, 128), (63, 130), (4096, 2), (4099, 2), (129, 65), (300, 40),
          (2050, 31), (700, 512), (90, 513), (33, 300), (1025, 1024)]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_layers(gpu, shape):
    """Per-column, per-row and scalar operands in every place of the binary ops, the unary ops, and a
    symbol used twice: tensors bit for bit, gradients bit for bit but for the sums over rows of more
    than 64 and over a row of more than 64 (each compared as the sum of its own terms)."""
    m = gpu.m
    r, w = shape
    vals = {"x": synth.normal(shape, 0, 1, 2200), "c": synth.uniform((1, w), 0.5, 1.5, 2201),
            "d": synth.normal((w,), 0, 0.5, 2202), "p": synth.uniform((r, 1), 0.5, 1.5, 2203), "k": np.array([1.5], np.float32)}
    nodes = [(OPS["MUL"], ["x", "c"], None, "h1"), (OPS["ADD"], ["h1", "d"], None, "h2"), (OPS["TANH"], ["h2"], None, "h3"),
             (OPS["MUL"], ["h3", "h3"], None, "h4"), (OPS["SUB"], ["p", "h4"], None, "h5"), (OPS["DIV"], ["h5", "p"], None, "h6"),
             (OPS["DIV"], ["h6", "c"], None, "h7"), (OPS["SIGMOID"], ["h7"], None, "h8"), (OPS["MUL"], ["h8", "k"], None, "h9"),
             (OPS["RELU"], ["h9"], None, "h10"), (OPS["EXP"], ["h10"], None, "h11")]
    trainable = ["x", "c", "d"] + (["p"] if r > 1 and w > 1 else [])
    ref = Graph(nodes, trainable)
    v = ref.forward(ORC, vals)
    seed = synth.normal(shape, 0, 1, 2204)
    gr = ref.backward(ORC, v, seed)
    g, syms, inputs = native_graph(m, nodes, vals, trainable, params=("c", "d", "p", "k"))
    g.out(syms["h11"])
    model = m.Model(g)
    for _ in range(2):  # the second pass from zeroed gradients again
        model.parameters.grads.set_zero()
        model.inference(*[vals[i] for i in inputs])
        model.backward(seed)
    P = model.parameters
    for n in ["h%d" % i for i in range(1, 12)]:
        assert_bitexact(P.tensors[syms[n]].to_numpy(), v[n], f"{shape} {n}")
    long_col, long_row = r > 64, w > 64
    # where a sum runs over more than 64 elements the oracle's order is another: there each element is
    # compared with the same nodes run one op call at a time on the device
    dev = Graph(nodes, trainable)
    dv = dev.forward(gpu, vals)
    gd = dev.backward(gpu, dv, seed)
    for n in ["x"] + ["h%d" % i for i in range(1, 11)]:  # no sum in them
        assert_bitexact(P.grads[syms[n]].to_numpy(), gr[n], f"{shape} grad {n}")
    if "p" in trainable:  # sums over a row
        assert_bitexact(P.grads[syms["p"]].to_numpy(), (gd if long_row else gr)["p"], f"{shape} grad p")
    if not long_col:
        for n in ("c", "d"):
            assert_bitexact(P.grads[syms[n]].to_numpy(), gr[n], f"{shape} grad {n}")
    # the longer sums over rows, each as the sum of its own terms (bit for bit the oracle's, above)
    terms = gr["h2"].astype(np.float64)
    assert_sum_close(P.grads[syms["d"]].to_numpy(), gr["d"], terms.sum(axis=0), f"{shape} grad d",
                     terms_abs=np.abs(terms).sum(axis=0))
    u1 = gr["h1"].astype(np.float64) * vals["x"].astype(np.float64)
    h6, c64 = v["h6"].astype(np.float64), vals["c"].astype(np.float64)
    u7 = -h6 / (c64 * c64) * gr["h7"].astype(np.float64)
    assert_sum_close(P.grads[syms["c"]].to_numpy(), gr["c"], (u1 + u7).sum(axis=0, keepdims=True), f"{shape} grad c",
                     terms_abs=(np.abs(u1) + np.abs(u7)).sum(axis=0, keepdims=True))


@pytest.mark.parametrize("shape", [(1, 2), (3, 64), (9, 65), (40, 168), (4, 2047), (700, 9), (5001, 60), (1024, 8), (1030, 7)],
                         ids=str)
def test_head(gpu, shape):
    """MAX, SUB, EXP, SUM, DIV, LOG, MUL, MEAN as programs: the gradient equals the same nodes run one
    op call at a time on the device, bit for bit; so does the loss."""
    m = gpu.m
    x, t = synth.normal(shape, 0, 2, 2210), synth.uniform(shape, 0, 1, 2211)
    synth.inject_ties(x, 1, 2212)
    from util import config5_nodes
    ref = Graph(config5_nodes(), ["logits"])
    v = ref.forward(gpu, {"logits": x, "onehot": t})
    gr = ref.backward(gpu, v, np.array([1.0], np.float32))
    g, syms, inputs = native_graph(m, config5_nodes(), {"logits": x, "onehot": t}, ["logits"])
    g.loss(syms["loss"])
    model = m.Model(g)
    loss = model.forward(*[{"logits": x, "onehot": t}[i] for i in inputs])
    model.backward()
    assert_bitexact(loss.to_numpy(), v["loss"], "loss")
    for n in ("max", "xm", "e", "s", "sm", "lp", "t"):
        assert_bitexact(model.parameters.tensors[syms[n]].to_numpy(), v[n], n)
        assert_bitexact(model.parameters.grads[syms[n]].to_numpy(), gr[n], f"grad {n}")
    assert_bitexact(model.parameters.grads[syms["logits"]].to_numpy(), gr["logits"], "grad logits")


@pytest.mark.parametrize("shape", [(5, 7), (128, 64), (1024, 8), (5001, 60)], ids=str)
def test_two_maxima_in_a_row(gpu, shape):
    """The gradients of two MAX nodes one after the other in a run, whose rows' maxima pass through the
    same shared memory: bit for bit what the nodes' own calls give."""
    m = gpu.m
    vals = {"a": synth.normal(shape, 0, 1, 2220), "b": synth.normal(shape, 3, 1, 2221)}
    synth.inject_ties(vals["a"], 1, 2222)
    nodes = [(OPS["MAX"], ["a"], 1, "ma"), (OPS["MAX"], ["b"], 1, "mb"),
             (OPS["MUL"], ["ma", "mb"], None, "h")]
    seed = synth.normal((shape[0], 1), 0, 1, 2223)
    ref = Graph(nodes, ["a", "b"])
    v = ref.forward(gpu, vals)
    gr = ref.backward(gpu, v, seed)
    g, syms, inputs = native_graph(m, nodes, vals, ["a", "b"])
    g.out(syms["h"])
    model = m.Model(g)
    model.inference(*[vals[i] for i in inputs])
    model.backward(seed)
    for n in ("a", "b"):
        assert_bitexact(model.parameters.grads[syms[n]].to_numpy(), gr[n], f"{shape} grad {n}")


@pytest.mark.parametrize("shape", [(4096, 2), (1025, 7), (1024, 8), (3000, 300)], ids=str)
def test_column_sums_do_not_depend_on_neighbours(gpu, shape):
    """The gradient of a per-column operand has the same bits whether a MAX stands in its run or the
    same row values come from outside: wherever a view has a program its sums go through it."""
    m = gpu.m
    vals = {"x": synth.normal(shape, 0, 1, 2230), "c": synth.uniform((1, shape[1]), 0.5, 1.5, 2231),
            "z": synth.normal(shape, 0, 1, 2232)}
    vals["p"] = ORC.forward(OPS["MAX"], vals["z"], axis=1)
    seed = synth.normal(shape, 0, 1, 2233)
    got = []
    for nodes, trainable in (([(OPS["MUL"], ["x", "c"], None, "h"), (OPS["MUL"], ["h", "p"], None, "out")], ["x", "c"]),
                             ([(OPS["MUL"], ["x", "c"], None, "h"), (OPS["MAX"], ["z"], 1, "mx"),
                               (OPS["MUL"], ["h", "mx"], None, "out")], ["x", "c", "z"])):
        use = {k: v for k, v in vals.items() if any(k in n[1] for n in nodes)}
        g, syms, inputs = native_graph(m, nodes, use, trainable, params=("c",))
        g.out(syms["out"])
        model = m.Model(g)
        model.inference(*[vals[i] for i in inputs])
        model.backward(seed)
        got.append(model.parameters.grads[syms["c"]].to_numpy())
    assert_bitexact(got[1], got[0], f"{shape} grad c")


@pytest.mark.parametrize("shape", [(4, 9), (32, 64), (64, 40), (70, 90), (90, 91), (8, 3)], ids=str)
@pytest.mark.parametrize("special", [False, True])
def test_whole_view_max(gpu, shape, special):
    """MAX over every element of a full and of a per-row tensor in one slab (up to 64 elements, below and
    above 2048), with LEAKYRELU and CLIP before it, on ordinary values and on +-0, NaN and infinities."""
    m = gpu.m
    r, w = shape
    x = synth.normal(shape, 0, 1, 2240)
    if special:
        x.reshape(-1)[:6] = [np.nan, np.inf, -np.inf, -0.0, 0.0, np.nan]
    p = np.abs(synth.normal((r, 1), 0, 1, 2241)) + np.float32(0.5)
    g = m.Graph()
    sx, sp = g.input(shape), g.input((r, 1))
    lk = g.op(m.OP.LEAKYRELU, sx, attributes={"negative_slope": 0.1})
    cl = g.op(m.OP.CLIP, lk, attributes={"min": -0.5, "max": 1.5})
    full = g.op(m.OP.MAX, cl)
    e = g.op(m.OP.EXP, sp)
    row = g.op(m.OP.MAX, e)
    out = g.op(m.OP.ADD, full, row)
    g.out(out)
    model = m.Model(g)
    model.inference(x, p)
    ref_l = ORC.forward(28, x, attrs={"negative_slope": 0.1})
    ref_c = ORC.forward(20, ref_l, attrs={"min": -0.5, "max": 1.5})
    T = model.parameters.tensors
    assert_bitexact(T[lk].to_numpy(), ref_l, "leakyrelu")
    assert_bitexact(T[cl].to_numpy(), ref_c, "clip")
    tx = gpu.T(ref_c)
    assert_bitexact(T[full].to_numpy(), m.tmax(tx).to_numpy(), "MAX of all as the op call")
    assert_bitexact(T[row].to_numpy(), m.tmax(T[e]).to_numpy(), "MAX of a per-row tensor as the op call")


def test_more_sums_than_one_program_holds(gpu):
    """A run with more per-column gradients than one program takes goes on in another."""
    m = gpu.m
    n, shape = 4200, (4100, 2)
    g = m.Graph()
    h = g.input(shape, trainable=True)
    syms = []
    for i in range(n):
        syms.append(g.param((1, 2), init=np.zeros(2, np.float32)))
        h = g.op(m.OP.ADD, h, syms[-1])
    g.out(h)
    model = m.Model(g)
    model.inference(synth.normal(shape, 0, 1, 2250))
    seed = np.ones(shape, np.float32)
    model.backward(seed)
    for i in (0, 1, n // 2, n - 4097, n - 4096, n - 1):
        assert_bitexact(model.parameters.grads[syms[i]].to_numpy(), np.full((1, 2), 4100, np.float32), f"grad {i}")


@pytest.mark.parametrize("fuse", [False, True])
@pytest.mark.parametrize("shape", [(64, 33), (700, 128)], ids=str)
def test_cut_inside_a_program(gpu, shape, fuse):
    """inference() ends inside a run, after an output in its middle: what lies before is written as by a whole
    pass, what lies behind is not; with and without fused bias + RELU pairs; a per-column parameter used
    in two layers of one run."""
    m = gpu.m
    w = shape[1]
    g = m.Graph()
    x = g.input(shape, trainable=True)
    c = g.param((1, w), init=synth.uniform((w,), 0.5, 1.5, 2260))
    b = g.param((1, w), init=synth.normal((w,), 0, 0.5, 2261))
    h1 = g.op(m.OP.RELU, g.op(m.OP.ADD, g.op(m.OP.MUL, x, c), b))
    h2 = g.op(m.OP.RELU, g.op(m.OP.ADD, g.op(m.OP.MUL, h1, c), b))
    g.out(h1)
    last = g.op(m.OP.TANH, h2)
    loss = g.op(m.OP.MEAN, last)
    g.loss(loss)
    model = m.Model(g, fuse_bias_relu=fuse)
    xv = synth.normal(shape, 0, 1, 2262)
    model.inference(xv)
    T = model.parameters.tensors
    got = T[h1].to_numpy()
    assert not T[last].to_numpy().any()
    model.forward(xv)
    assert_bitexact(T[h1].to_numpy(), got, "output of the cut")
    model.backward()
    cv, bv = T[c].to_numpy(), T[b].to_numpy()
    v64 = {}
    v64["h1"] = np.maximum(xv.astype(np.float64) * cv + bv, 0)
    v64["h2"] = np.maximum(v64["h1"] * cv + bv, 0)
    u2 = (1 - np.tanh(v64["h2"]) ** 2) / xv.size * (v64["h2"] > 0)
    u1 = u2 * cv * (v64["h1"] > 0)
    G = model.parameters.grads
    for sym, terms in ((c, u2 * v64["h1"] + u1 * xv), (b, u2 + u1)):
        # 1e-5 of the sum of |terms|: a few float32 roundings of each term and its sum's order
        err = np.abs(G[sym].to_numpy() - terms.sum(axis=0, keepdims=True))
        assert (err <= 1e-5 * np.abs(terms).sum(axis=0, keepdims=True) + 1e-12).all(), err.max()
