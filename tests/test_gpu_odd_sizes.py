"""Rows and columns of every length modulo 4 and at every 4-byte alignment: the kernels move them as
unaligned quads, the last few elements of a line apart. Lines at the edges of the kernels' ranges
against the oracle, and views of a larger tensor (offsets of 1-3 floats) against the same values
at an aligned address."""
import numpy as np
import pytest

from mantle_amd import synth
from util import O, OPS, GpuEngine, Graph, OracleEngine, assert_bitexact, assert_sum_close, softmax_nodes

pytestmark = pytest.mark.gpu
ORC = OracleEngine()
SUM, MEAN, MAX = OPS["SUM"], OPS["MEAN"], OPS["MAX"]


@pytest.fixture(scope="module")
def gpu():
    return GpuEngine()


@pytest.fixture(autouse=True)
def _nelts():
    O.set_nelts(32)
    yield


def view(gpu, a, off):
    """`a` at `off` floats past an aligned address, with nothing after its last element's quad."""
    buf = gpu.T(np.concatenate([np.full(off, 7.0, np.float32), np.asarray(a, np.float32).reshape(-1)]))
    return gpu.m.Tensor(gpu.m.TensorShape(*np.asarray(a).shape), _ptr=buf.ptr + 4 * off, _owner=buf)


def reductions_match(gpu, shape, axis, off=0):
    """SUM, MEAN, MAX forward and backward, and tstd, of one shape against the oracle; x holds
    ties, the gradient -0, +0 and NaN (the sums go by the condition of their terms)."""
    m = gpu.m
    x = synth.normal(shape, 0, 1, 2100)
    if shape[axis] > 2:
        synth.inject_ties(x, axis, 2101)
    red = tuple(1 if i == axis else d for i, d in enumerate(shape))
    ug = synth.normal(red, 0, 1, 2102)
    g0 = synth.normal(shape, 0, 1, 2103).reshape(-1)
    g0[::3], g0[1::7], g0[2::11] = np.float32(-0.0), np.float32(0.0), np.float32(np.nan)
    g0 = g0.reshape(shape)
    tx, tu = view(gpu, x, off), view(gpu, ug, off)
    x64 = x.astype(np.float64)
    for op, ex, mag in ((SUM, x64.sum(axis=axis, keepdims=True), np.abs(x64).sum(axis=axis, keepdims=True)),
                        (MEAN, x64.mean(axis=axis, keepdims=True), np.abs(x64).mean(axis=axis, keepdims=True)),
                        (MAX, None, None)):
        res, g = view(gpu, np.zeros(red, np.float32), off), view(gpu, g0, off)
        m.forward_op(op, res, tx, attributes={"axis": axis})
        ref = ORC.forward(op, x, axis=axis)
        if op == MAX:
            assert np.array_equal(res.to_numpy(), ref)  # equal as floats: a zero tie's sign follows the order
        else:
            assert_sum_close(res.to_numpy(), ref, ex, f"{shape} axis {axis} op {op}", terms_abs=mag)
        m.backward_op(0, op, tu, tx, None, g, attributes={"axis": axis})
        assert_bitexact(g.to_numpy(), ORC.backward(0, op, ug, x, axis=axis, grad=g0), f"{shape} axis {axis} op {op} bwd")
    assert_sum_close(m.tstd(tx, axis).to_numpy(), ORC.tstd(x, axis), x64.std(axis=axis, keepdims=True),
                     f"tstd {shape} axis {axis}")


@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("b", [1, 2, 5, 33, 65, 67, 255, 257, 1021, 1023, 1026, 2047, 2049, 2051, 4095, 8191, 16383,
                               16385, 20479])
def test_rows(gpu, b, off):
    """Last-axis lines: the short-row tiles, one wavefront, rows in registers and chunks of 2048."""
    reductions_match(gpu, (5, b), 1, off)


@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("b", [4, 32, 36, 64, 256, 260, 1024, 2048, 4096, 4100, 8192, 16384])
def test_rows_of_whole_quads(gpu, b, off):
    """Last-axis lines of whole quads, at any address: the row kernels' variants without selects, and
    short rows at an unaligned address in two passes."""
    reductions_match(gpu, (5, b), 1, off)


@pytest.mark.parametrize("off", [0, 2])
@pytest.mark.parametrize("b", [65, 66, 67, 68, 127, 250, 253, 255, 256, 257, 258, 259, 260, 511, 770, 771, 772, 773, 775,
                               1022, 1025, 2045])
def test_rows_by_wavefront(gpu, b, off):
    """A row per wavefront at the edges of its quad counts (64, 192 and the groups of 256), with every
    length modulo 4, in the order of its sums: quads lane, lane + 64, ... in groups of four, the last
    elements after them, then a butterfly."""
    def row_sum(x):
        f, nq = np.float32, b // 4
        a4 = np.zeros((64, 4, 4), f)
        for lane in range(64):
            q = lane
            while q + 192 < nq:
                for u in range(4):
                    a4[lane, u] += x[4 * (q + 64 * u):4 * (q + 64 * u) + 4]
                q += 256
            while q < nq:
                a4[lane, 0] += x[4 * q:4 * q + 4]
                q += 64
            if q == nq:
                a4[lane, 0, :b % 4] += x[4 * nq:b]
        v = np.zeros(64, f)
        for g in a4.reshape(64, 16).T:
            v = v + g
        for k in (32, 16, 8, 4, 2, 1):
            v = v + v[np.arange(64) ^ k]
        return v[0]

    x = synth.normal((6, b), 0, 1, 2115)
    res = view(gpu, np.zeros((6, 1), np.float32), 0)
    gpu.m.forward_op(SUM, res, view(gpu, x, off), attributes={"axis": 1})
    assert_bitexact(res.to_numpy()[:, 0], np.array([row_sum(r) for r in x], np.float32), f"SUM over {b}")
    x[1, ::3], x[2, -1], x[3] = np.nan, np.inf, -np.inf
    gpu.m.forward_op(MAX, res, view(gpu, x, off), attributes={"axis": 1})
    got = res.to_numpy()[:, 0]
    for r in (0, 2, 4, 5):
        assert got[r] == x[r].max(), r
    assert got[3] == -np.finfo(np.float32).max  # MAX starts at -FLT_MAX


@pytest.mark.parametrize("n", [262145, 262146 + 4 * 2048, 1 << 20, (1 << 20) + 3])
def test_every_element(gpu, n):
    """All elements as one row of chunks, whose last one is ragged."""
    x = synth.normal((n,), 0, 1, 2110)
    x[n // 2] = x[n - 1] = np.float32(9.0)
    x64 = x.astype(np.float64)
    assert_sum_close(gpu.forward(SUM, x), ORC.forward(SUM, x), np.array([x64.sum()]), terms_abs=np.array([np.abs(x64).sum()]))
    assert np.array_equal(gpu.forward(MAX, x), ORC.forward(MAX, x))
    ug = np.array([0.75], np.float32)
    assert_bitexact(gpu.backward(0, MAX, ug, x), ORC.backward(0, MAX, ug, x), "MAX bwd")
    assert_sum_close(gpu.tstd(x), ORC.tstd(x), np.array([x64.std()]), "tstd")


@pytest.mark.parametrize("off", [0, 2])
@pytest.mark.parametrize("rows,classes", [(1, 65), (2, 66), (3, 67), (9, 127), (8, 128), (5, 129), (3, 131), (4, 255),
                                          (5, 256), (5, 257), (3, 511), (2, 513), (7, 832), (3, 836), (1, 1021),
                                          (2, 1022), (3, 1023), (2, 1024), (1, 1025), (2, 2045), (1, 2047)])
def test_softmax_rows(gpu, rows, classes, off):
    """Fused Softmax at the class counts where the lanes per row and the elements per lane change,
    and at the tensor's last row, whose last quad would leave it: bit for bit the op-by-op graph."""
    m = gpu.m
    x, gout = synth.normal((rows, classes), 0, 2, 2120), synth.normal((rows, classes), 0, 1, 2121)
    g0 = synth.normal((rows, classes), 0, 1, 2122)
    g = Graph(softmax_nodes("x", 1), ["x"])
    v = g.forward(gpu, {"x": x})
    gr = g.backward(gpu, v, seed=gout, init={"x": g0})
    out, tg, tx = view(gpu, np.zeros_like(x), off), view(gpu, g0, off), view(gpu, x, off)
    m.softmax_forward(out, tx)
    m.softmax_backward(tg, tx, view(gpu, gout, off))
    assert_bitexact(out.to_numpy(), v["sm"], "softmax")
    assert_bitexact(tg.to_numpy(), gr["x"], "softmax backward")


@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("shape", [(1, 70, 3), (1, 5000, 2), (2, 33, 5), (5, 1, 7), (7, 17, 6), (3, 100, 127),
                                   (2, 65, 129), (1, 300, 1023), (2, 129, 1025), (1, 2100, 1026), (1, 9, 4097),
                                   (40, 64, 9), (1, 513, 4)], ids=str)
def test_columns(gpu, shape, off):
    """Strided axes: single columns, column quads whose last one overlaps the one before, strips
    and wide forms, in one split and in several."""
    reductions_match(gpu, shape, 1, off)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("shape", [(1, 7, 4), (3, 8, 5), (2, 9, 19), (1, 15, 20), (4, 17, 1030), (2, 31, 1028), (2100, 3, 129),
                                   (2100, 9, 132), (2500, 17, 33), (2500, 40, 36), (1, 1100, 9), (40, 33, 2)], ids=str)
def test_columns_in_every_form(gpu, shape, off):
    """Strided axes at the edges of the forms' rules, with rows left over from the eight (four, two) in
    flight."""
    reductions_match(gpu, shape, 1, off)


@pytest.mark.parametrize("off", [0, 3])
@pytest.mark.parametrize("shape", [(1, 8200, 2051), (2, 4100, 2049), (300, 1800, 33), (1, 16400, 1026), (1, 420000, 41)], ids=str)
def test_max_backward_routes_by_indices(gpu, shape, off):
    """MAX backward over columns large enough to route by the splits' indices, of widths whose last quad
    overlaps the one before: ties inside a split and across splits, a gradient of -0, +0 and NaN."""
    m = gpu.m
    x = synth.normal(shape, 0, 1, 2300)
    a, b, c = shape
    x[:, 5, ::3] = x[:, b // 2, ::3] = x[:, b - 1, ::3] = np.float32(9.0)  # across splits
    x[:, 7, 1::5] = x[:, 8, 1::5] = np.float32(8.0)                         # inside one
    ug, g0 = synth.normal((a, 1, c), 0, 1, 2301), synth.normal(shape, 0, 1, 2302).reshape(-1)
    g0[::3], g0[1::7], g0[2::11] = np.float32(-0.0), np.float32(0.0), np.float32(np.nan)
    g0 = g0.reshape(shape)
    g = view(gpu, g0, off)
    m.backward_op(0, MAX, view(gpu, ug, off), view(gpu, x, off), None, g, attributes={"axis": 1})
    assert_bitexact(g.to_numpy(), ORC.backward(0, MAX, ug, x, axis=1, grad=g0), f"{shape} off {off}")


@pytest.mark.parametrize("op", ["SUB", "MUL", "DIV"])
@pytest.mark.parametrize("shape,bshape", [((300, 1001), (1, 1001)), ((70, 5), (1, 5)), ((129, 2), (1, 2)),
                                          ((4099, 130), (130,)), ((3, 200, 67), (3, 1, 67)), ((1000, 3), (3,))],
                         ids=str)
def test_unbroadcast_columns(gpu, op, shape, bshape):
    """The gradient of an operand that repeats over rows, accumulated into a nonzero gradient."""
    x, b = synth.normal(shape, 0, 1, 2130), synth.uniform(bshape, 0.5, 2, 2131)
    ug, g0 = synth.normal(shape, 0, 1, 2132), synth.normal(bshape, 0, 1, 2133)
    x64, b64, u64 = (v.astype(np.float64) for v in (x, b, ug))
    rg = {"SUB": -u64 + 0 * b64, "MUL": u64 * x64, "DIV": -x64 / (b64 * b64) * u64}[op]
    lead = rg.ndim - len(bshape)
    axes = tuple(range(lead)) + tuple(i + lead for i, d in enumerate(bshape) if d == 1 and shape[i + lead] > 1)
    total = lambda v: v.sum(axis=axes, keepdims=True).reshape(bshape)  # noqa: E731
    assert_sum_close(gpu.backward(1, OPS[op], ug, x, b, grad=g0), O.backward_op(1, OPS[op], ug, x, b, grad=g0),
                     total(rg) + g0, f"{op} {shape}", terms_abs=total(np.abs(rg)) + np.abs(g0))


BCAST_FORMS = [((3, 5, 7), (1, 5, 1)), ((3, 5, 7), (3, 1, 7)), ((3, 5, 7), (1, 1, 7)), ((3, 5, 7), (3, 5, 1)),
               ((2, 3, 4), (2, 1, 4)), ((4, 1, 9), (1, 6, 1)), ((4, 1, 9), (1, 6, 9)), ((4, 6, 1), (1, 1, 11)),
               ((129, 5), (5,)), ((17, 9, 13), (9, 1)), ((5, 3, 131), (5, 1, 131)), ((2, 33, 729), (1, 33, 1)),
               ((1, 64, 6), (5, 1, 6)), ((7, 2, 3, 5), (7, 1, 3, 5)), ((6, 1, 5), (1, 4, 5)),
               ((1001, 2), (2,)), ((33, 3), (3,)), ((5, 7, 3), (7, 1)), ((5, 7, 2), (5, 1, 2)), ((5, 7, 3), (5, 7, 1)), ((9, 6, 2), (6, 2))]


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("s1,s2", BCAST_FORMS, ids=str)
def test_broadcast_forms(gpu, s1, s2, off):
    """A broadcast operand in either place, constant or contiguous inside a row whose length is not
    (or is) a multiple of 4, both operands broadcast, and their gradients; the broadcast operand
    also at an unaligned address. Element values are single operations: bit for bit."""
    m = gpu.m
    a, b = synth.normal(s1, 0, 1, 2140), synth.uniform(s2, 0.5, 2, 2141)
    for x, y, x_off, y_off in ((a, b, 0, off), (b, a, off, 0)):
        tx, ty = view(gpu, x, x_off), view(gpu, y, y_off)
        so = np.broadcast_shapes(x.shape, y.shape)
        ug, g0 = synth.normal(so, 0, 1, 2142), synth.normal(x.shape, 0, 1, 2143)
        for op in (OPS["SUB"], OPS["MUL"], OPS["DIV"]):
            res = m.Tensor(m.TensorShape(*so))
            m.forward_op(op, res, tx, ty)
            assert_bitexact(res.to_numpy(), ORC.forward(op, x, y), f"{s1} {s2} op {op}")
            for i, (p, q) in enumerate(((x, y), (y, x))):
                g0 = synth.normal(p.shape, 0, 1, 2144 + i)
                got = gpu.backward(i, op, ug, x, y, grad=g0)
                if p.shape == so:  # no sum: the same single operations
                    assert_bitexact(got, ORC.backward(i, op, ug, x, y, grad=g0), f"{s1} {s2} op {op} id {i}")


@pytest.mark.parametrize("shape,axis", [((6, 3, 7), 1), ((9, 2, 131), 1), ((5, 3, 2, 9), 1), ((2, 30, 1001), 1), ((7, 9), 0)],
                         ids=str)
def test_reduce_backward_short_axes(gpu, shape, axis):
    """Reductions over an axis too short to split: the line operands of SUM, MEAN and MAX backward
    broadcast over it."""
    reductions_match(gpu, shape, axis)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("shape", [(3, 5, 64), (2, 3, 65), (70, 3, 67), (5, 2, 729), (1, 4, 4099), (2, 2, 4102), (3, 1, 130)],
                         ids=str)
def test_channel_gradients(gpu, shape, off):
    """The gradient of a per-channel operand [1, C, 1] over planes of every length modulo 4, one and
    several chunks a plane, in either place of the binary ops; ug also at an unaligned address."""
    m = gpu.m
    x, b = synth.uniform(shape, 0.5, 2, 2150), synth.uniform((1, shape[1], 1), 0.5, 2, 2151)
    ug, g0 = synth.normal(shape, 0, 1, 2152), synth.normal((1, shape[1], 1), 0, 1, 2153)
    x64, b64, u64 = (v.astype(np.float64) for v in (x, b, ug))
    for name, i, rg in (("ADD", 1, u64), ("SUB", 1, -u64), ("SUB", 0, u64), ("MUL", 0, u64 * x64), ("MUL", 1, u64 * x64),
                        ("DIV", 0, u64 / x64), ("DIV", 1, -x64 / (b64 * b64) * u64)):
        t1, t2 = (b, x) if i == 0 else (x, b)
        g = gpu.T(g0)
        m.backward_op(i, OPS[name], view(gpu, ug, off), gpu.T(t1), gpu.T(t2), g)
        ref = O.backward_op(i, OPS[name], ug, t1, t2, grad=g0)
        assert_sum_close(g.to_numpy(), ref, rg.sum(axis=(0, 2), keepdims=True) + g0, f"{name} id {i} {shape}",
                         terms_abs=np.abs(rg).sum(axis=(0, 2), keepdims=True) + np.abs(g0))


@pytest.mark.parametrize("rows,cols", [(65, 4), (64, 8), (70, 5), (300, 33), (4500, 6), (130, 511), (97, 512), (66, 1030), (2300, 530),
                                       (1301, 302),
                                       (129, 1027)])
def test_linear_bias_relu(gpu, rows, cols):
    """Bias + RELU over [rows, features], one pass each way: outputs and per-element gradients bit for
    bit the op-by-op calls', the bias gradient in the sum class; with and without the kept gradients."""
    m = gpu.m
    x, b = synth.normal((rows, cols), 0, 1, 2160), synth.normal((1, cols), 0, 0.5, 2161)
    x[::3] = 0.0
    b[:, ::2] = -0.0
    ug, g0, gb0 = synth.normal((rows, cols), 0, 1, 2162), synth.normal((rows, cols), 0, 1, 2163), synth.normal((1, cols), 0, 1, 2164)
    y, r = gpu.T(np.zeros_like(x)), gpu.T(np.zeros_like(x))
    m.bias_relu_forward(y, r, gpu.T(x), gpu.T(b))
    yr = ORC.forward(OPS["ADD"], x, b)
    assert_bitexact(y.to_numpy(), yr, "y")
    assert_bitexact(r.to_numpy(), ORC.forward(OPS["RELU"], yr), "r")
    for keep_y, keep_x in ((True, True), (False, True), (True, False), (False, False)):
        gy = ORC.backward(0, OPS["RELU"], ug, yr, grad=g0 if keep_y else np.zeros_like(x))
        ty, tx, tb = gpu.T(g0), gpu.T(g0), gpu.T(gb0)
        m.bias_relu_backward(gpu.T(ug), y, b.shape, tx if keep_x else None, tb, ty if keep_y else None)
        if keep_y:
            assert_bitexact(ty.to_numpy(), gy, "grad y")
        if keep_x:
            assert_bitexact(tx.to_numpy(), ORC.backward(0, OPS["ADD"], gy, x, b, grad=g0), "grad x")
        g64 = gy.astype(np.float64)
        assert_sum_close(tb.to_numpy(), O.backward_op(1, OPS["ADD"], gy, x, b, grad=gb0),
                         g64.sum(axis=0, keepdims=True) + gb0, "grad bias",
                         terms_abs=np.abs(g64).sum(axis=0, keepdims=True) + np.abs(gb0))
