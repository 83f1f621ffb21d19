// mh_model.hip -- Mantle's Graph builder (mantle/autograd/graph.mojo:33-217) and Model
// executor (mantle/nn/model.mojo:55-340) with its two Collections (tensors and grads,
// mantle/autograd/collection.mojo:24-224, mantle/nn/parameters.mojo) held in device memory.
//
// A graph records symbols (inputs, parameters, node outputs) and nodes in creation order,
// which is a topological order (graph.mojo:448-451). A model built from it places every
// symbol in one device arena and every trainable symbol's gradient in a second one, each
// tensor on a 256-byte boundary so the float4 paths apply, and runs forward / backward as
// back-to-back launches on the library stream with one synchronisation at the end (none
// under MH_INIT_ASYNC). Inputs enter by copy into their slots, as Collection.__setitem__
// does (collection.mojo:202-209); everything else stays on the device.
//
// Optional fusion: an ADD whose output feeds only the RELU node right after it runs as the
// fused bias + RELU kernels (MH_MODEL_FUSE_BIAS_RELU), and the node runs of nn.Softmax,
// nn.LogSoftmax, CrossEntropyLoss and the Softmax -> LOG -> MUL -> MEAN head run as the
// row-fused kernels (MH_MODEL_FUSE_ROWS). Runs of nodes over one [R, W] view whose tensors are
// small, or that would re-read from memory what they just wrote, go as one launch
// (mh_program.hip), planned when the model is made. Every slot that these write holds the bits of
// the op-by-op execution, except the gradients that are sums over more than 64 rows of a per-column
// operand (a bias): those are summed in an order of the fused kernel's or the program's own, which
// depends on the flags and the view but not on the nodes around.
// mh_model_capture records a pass (forward, backward, or zero_grad + forward + backward) as
// one HIP graph that mh_model_replay launches. While a captured graph exists, a library
// buffer that grows is retired rather than freed, so the addresses the graph holds stay
// valid until the graph is released or the library shuts down (a replay after mh_shutdown is
// refused).
#include <new>
#include <unordered_map>
#include <vector>

#include "mh_program.h"

struct mh_graph {
    struct Sym {
        mh_shape shape;
        int trainable;
        int kind;          // MH_SYM_INPUT / MH_SYM_PARAM / MH_SYM_NODE
        int64_t init_off;  // parameter data in init_data, or -1 (zero-initialised)
    };
    struct Node {
        int op;
        int nin;
        int32_t in[3];
        int32_t out;
        mh_attrs attrs;
    };
    std::vector<Sym> syms;
    std::vector<float> init_data;
    std::vector<int32_t> inputs, params, outputs;
    int32_t loss = -1;
    std::vector<Node> nodes;
};

struct mh_model {
    mh_graph g;
    uint64_t flags = 0;
    float* arena = nullptr;
    float* grad_arena = nullptr;
    size_t arena_floats = 0, grad_floats = 0;
    std::vector<float*> t;  // per symbol: its tensor slot
    std::vector<float*> gr;  // per symbol: its gradient slot (nullptr if not trainable)
    int32_t n_inference = -1;
    size_t param_span = 0;  // floats of the trainable-parameter span at the start of both arenas
    std::vector<int> fuse;  // per node: kFuseAdd / kFuseRelu (bias + RELU), kFuseRow (row group)
    struct RowGroup {
        int graph;  // 0 head (Softmax, LOG, MUL, MEAN), 1 cross entropy, 2 Softmax, 3 LogSoftmax
        int first, last;
        int32_t x, target, out;
        int64_t rows, K;
        float scale;  // cross entropy: the graph scalar of its last MUL
    };
    std::vector<RowGroup> rows;
    std::vector<int> row_of;  // per node: its RowGroup, or -1
    struct Segment {
        int first, last;  // nodes, in creation order
        mh::ProgRun run;
    };
    std::vector<Segment> fseg, bseg;          // forward and backward programs
    std::vector<int> fseg_of, bseg_of;        // per node: its Segment, or -1
    void* prog_mem = nullptr;                 // their instructions and sums
    float* prog_part = nullptr;               // partials of one program at a time
    hipGraphExec_t graph[3] = {nullptr, nullptr, nullptr};  // captured passes (MH_PASS_FORWARD / _BACKWARD / _STEP)
    uint64_t graph_epoch[3] = {0, 0, 0};                     // the mh_init epoch each was captured in
};

namespace mh {

static int op_arity(int op) {
    switch (op) {
        case MH_ADD: case MH_SUB: case MH_MUL: case MH_DIV: case MH_POW: return 2;
        case MH_EXP: case MH_LOG: case MH_SIGMOID: case MH_RELU: case MH_TANH:
        case MH_SUM: case MH_MEAN: case MH_MAX: case MH_CLIP: case MH_LEAKYRELU: return 1;
        case MH_FMA: return 3;
        default: return 0;
    }
}

static int axis_of(const mh_attrs& a) { return (a.flags & MH_ATTR_AXIS) ? a.axis : -1; }
static bool is_binary(int op) { return op >= MH_ADD && op <= MH_DIV; }
static bool is_unary(int op) {
    return op == MH_EXP || op == MH_LOG || op == MH_SIGMOID || op == MH_RELU || op == MH_TANH;
}
static bool is_reduce(int op) { return op == MH_SUM || op == MH_MEAN || op == MH_MAX; }
static float clip_lo(const mh_attrs& a) { return (a.flags & MH_ATTR_MIN) ? a.min_val : -3.40282347e38f; }
static float clip_hi(const mh_attrs& a) { return (a.flags & MH_ATTR_MAX) ? a.max_val : 3.40282347e38f; }

// static_result_shape (ops.mojo:104-218) for the ops of this path.
static int result_shape(const mh_graph& g, int op, int nin, const int32_t* in, const mh_attrs& at, mh_shape* out) {
    const mh_shape& s1 = g.syms[in[0]].shape;
    if (is_binary(op)) return broadcast_shapes(s1, g.syms[in[1]].shape, out);
    if (op == MH_POW) {
        if (!is_scalar_shape(g.syms[in[1]].shape))
            return fail(MH_ERR_SHAPE, "POW: the exponent must be a shape-(1) symbol (basics.mojo:317)");
        *out = s1;
        return MH_OK;
    }
    if (is_reduce(op)) {
        const int ax = axis_of(at);
        if (ax < -1 || ax >= s1.rank) return fail(MH_ERR_INVALID, "reduce: axis %d outside [-1, %d)", ax, s1.rank);
        *out = reduced_shape(s1, ax);
        return MH_OK;
    }
    if (op == MH_FMA) {
        if (!shape_eq(s1, g.syms[in[1]].shape) || !shape_eq(s1, g.syms[in[2]].shape))
            return fail(MH_ERR_SHAPE, "FMA: the three operands must have one shape (basics.mojo:759-766)");
    }
    if (op == MH_LEAKYRELU && !(at.flags & MH_ATTR_NEGATIVE_SLOPE))
        return fail(MH_ERR_INVALID, "LEAKYRELU needs the negative_slope attribute (mlops.mojo:145)");
    (void)nin;
    *out = s1;
    return MH_OK;
}

static int add_symbol(mh_graph* g, const mh_shape& s, int trainable, int kind, int32_t* sym) {
    MH_TRY(check_shape(s, "symbol"));
    if (g->syms.size() >= 0x7fffffff) return fail(MH_ERR_INVALID, "too many symbols");
    mh_graph::Sym y;
    y.shape = s;
    y.trainable = trainable ? 1 : 0;
    y.kind = kind;
    y.init_off = -1;
    g->syms.push_back(y);
    *sym = (int32_t)(g->syms.size() - 1);
    return MH_OK;
}

static int check_sym(const mh_graph* g, int32_t sym) {
    if (sym < 0 || (size_t)sym >= g->syms.size()) return fail(MH_ERR_INVALID, "unknown symbol %d", sym);
    return MH_OK;
}

static size_t slot_floats(const mh_shape& s) {
    const size_t n = (size_t)numel(s);
    return (n + 63) & ~(size_t)63;  // 256-byte slots
}

// Sets MH_INIT_ASYNC for the ops of one model pass; synchronises once at the end when the
// caller did not ask for asynchronous calls.
struct PassScope {
    uint64_t saved;
    PassScope() : saved(ctx().flags) { ctx().flags |= MH_INIT_ASYNC; }
    ~PassScope() { ctx().flags = saved; }
    int end(const char* what) {
        ctx().flags = saved;
        return finish(what);
    }
};

static int copy_in(float* dst, const float* src, size_t n, int where) {
    if (n == 0) return MH_OK;
    if (!src) return fail(MH_ERR_NULL, "null input tensor");
    const hipMemcpyKind k = where == MH_FROM_HOST ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice;
    MH_HIP(hipMemcpyAsync(dst, src, n * sizeof(float), k, ctx().stream));
    return MH_OK;
}

// n_inference_nodes (model.mojo:39-48): one past the last node that writes a graph output.
static int32_t inference_nodes(const mh_graph& g) {
    for (int32_t i = (int32_t)g.nodes.size() - 1; i >= 0; --i)
        for (int32_t o : g.outputs)
            if (g.nodes[i].out == o) return i + 1;
    return -1;
}

constexpr int kFuseAdd = 1, kFuseRelu = 2, kFuseRow = 3;
constexpr int64_t kRowMaxClasses = 2047;  // the fused row kernels' limit

// Row groups (MH_MODEL_FUSE_ROWS): consecutive nodes that nn.Softmax / nn.LogSoftmax /
// nn.CrossEntropyLoss emit (activations.mojo:74-108, loss.mojo:45-61), or the config-5 head
// (Softmax, LOG, MUL by a target, MEAN), over the last axis, whose intermediates are read by
// the group alone and are neither graph outputs nor the loss.
static void plan_row_groups(mh_model* m) {
    const mh_graph& g = m->g;
    const size_t nn = g.nodes.size();
    std::vector<std::vector<int>> users(g.syms.size());
    for (size_t j = 0; j < nn; ++j)
        for (int k = 0; k < g.nodes[j].nin; ++k) users[g.nodes[j].in[k]].push_back((int)j);
    auto exported = [&](int32_t sym) {
        if (g.loss == sym) return true;
        for (int32_t o : g.outputs)
            if (o == sym) return true;
        return false;
    };
    // every reader of `sym` lies in [first, last], and it is not exported
    auto local = [&](int32_t sym, int first, int last) {
        if (exported(sym)) return false;
        for (int j : users[sym])
            if (j < first || j > last) return false;
        return true;
    };
    auto node_is = [&](size_t j, int op) { return j < nn && g.nodes[j].op == op && m->fuse[j] == 0; };
    auto axis_last = [&](const mh_graph::Node& nd, const mh_shape& s) {
        return (nd.attrs.flags & MH_ATTR_AXIS) && nd.attrs.axis == s.rank - 1;
    };
    for (size_t i = 0; i + 4 < nn; ++i) {
        const mh_graph::Node& n0 = g.nodes[i];
        if (!node_is(i, MH_MAX)) continue;
        const int32_t x = n0.in[0];
        const mh_shape& sx = g.syms[x].shape;
        if (!axis_last(n0, sx)) continue;
        const int64_t K = sx.dims[sx.rank - 1];
        if (K < 1 || K > kRowMaxClasses) continue;
        const mh_graph::Node &n1 = g.nodes[i + 1], &n2 = g.nodes[i + 2], &n3 = g.nodes[i + 3];
        if (!node_is(i + 1, MH_SUB) || n1.in[0] != x || n1.in[1] != n0.out) continue;
        if (!node_is(i + 2, MH_EXP) || n2.in[0] != n1.out) continue;
        if (!node_is(i + 3, MH_SUM) || n3.in[0] != n2.out || !axis_last(n3, sx)) continue;
        mh_model::RowGroup rg{};
        rg.x = x;
        rg.rows = numel(sx) / K;
        rg.K = K;
        rg.first = (int)i;
        const mh_graph::Node& n4 = g.nodes[i + 4];
        int32_t core_out;
        if (node_is(i + 4, MH_DIV) && n4.in[0] == n2.out && n4.in[1] == n3.out) {
            rg.graph = 2;  // Softmax
            rg.last = (int)i + 4;
        } else if (node_is(i + 4, MH_LOG) && n4.in[0] == n3.out && node_is(i + 5, MH_SUB) &&
                   g.nodes[i + 5].in[0] == n1.out && g.nodes[i + 5].in[1] == n4.out) {
            rg.graph = 3;  // LogSoftmax
            rg.last = (int)i + 5;
        } else {
            continue;
        }
        core_out = g.nodes[rg.last].out;
        rg.out = core_out;
        // a loss on top: the head (Softmax, LOG, MUL(target), MEAN) or the cross entropy
        // (LogSoftmax, MUL(target), SUM, MUL(scalar)), target not trainable, x of rank 2 for
        // the cross entropy (its axis 1)
        auto mul_target = [&](size_t j, int32_t v, int32_t* t) {
            if (!node_is(j, MH_MUL)) return false;
            const mh_graph::Node& nd = g.nodes[j];
            const int32_t o = nd.in[0] == v ? nd.in[1] : nd.in[1] == v ? nd.in[0] : -1;
            if (o < 0 || o == v || g.syms[o].trainable || !shape_eq(g.syms[o].shape, sx)) return false;
            *t = o;
            return true;
        };
        int32_t t = -1;
        const size_t L = (size_t)rg.last;
        if (rg.graph == 2 && node_is(L + 1, MH_LOG) && g.nodes[L + 1].in[0] == core_out &&
            mul_target(L + 2, g.nodes[L + 1].out, &t) && node_is(L + 3, MH_MEAN) &&
            g.nodes[L + 3].in[0] == g.nodes[L + 2].out && !(g.nodes[L + 3].attrs.flags & MH_ATTR_AXIS)) {
            mh_model::RowGroup h = rg;
            h.graph = 0;
            h.last = (int)L + 3;
            h.target = t;
            h.out = g.nodes[L + 3].out;
            if (local(core_out, h.first, h.last) && local(g.nodes[L + 1].out, h.first, h.last) &&
                local(g.nodes[L + 2].out, h.first, h.last))
                rg = h;
        } else if (rg.graph == 3 && sx.rank == 2 && mul_target(L + 1, core_out, &t) && node_is(L + 2, MH_SUM) &&
                   g.nodes[L + 2].in[0] == g.nodes[L + 1].out && !(g.nodes[L + 2].attrs.flags & MH_ATTR_AXIS) &&
                   node_is(L + 3, MH_MUL) && g.nodes[L + 3].in[0] == g.nodes[L + 2].out) {
            const int32_t c = g.nodes[L + 3].in[1];
            const mh_graph::Sym& cs = g.syms[c];
            if (cs.kind == MH_SYM_PARAM && !cs.trainable && cs.init_off >= 0 && is_scalar_shape(cs.shape)) {
                mh_model::RowGroup h = rg;
                h.graph = 1;
                h.last = (int)L + 3;
                h.target = t;
                h.out = g.nodes[L + 3].out;
                h.scale = g.init_data[(size_t)cs.init_off];
                if (local(core_out, h.first, h.last) && local(g.nodes[L + 1].out, h.first, h.last) &&
                    local(g.nodes[L + 2].out, h.first, h.last))
                    rg = h;
            }
        }
        // the core's intermediates: MAX, SUB, EXP, SUM (and LOG of LogSoftmax) outputs
        bool ok = true;
        for (int j = rg.first; j < (rg.graph == 3 || rg.graph == 1 ? rg.first + 5 : rg.first + 4) && ok; ++j)
            ok = local(g.nodes[j].out, rg.first, rg.last);
        if (!ok) continue;
        const int id = (int)m->rows.size();
        m->rows.push_back(rg);
        for (int j = rg.first; j <= rg.last; ++j) {
            m->fuse[j] = kFuseRow;
            m->row_of[j] = id;
        }
        i = (size_t)rg.last;
    }
}

static void plan_fusion(mh_model* m) {
    const mh_graph& g = m->g;
    m->fuse.assign(g.nodes.size(), 0);
    m->row_of.assign(g.nodes.size(), -1);
    m->rows.clear();
    if (m->flags & MH_MODEL_FUSE_ROWS) plan_row_groups(m);
    if (!(m->flags & MH_MODEL_FUSE_BIAS_RELU)) return;
    for (size_t i = 0; i + 1 < g.nodes.size(); ++i) {
        const mh_graph::Node& a = g.nodes[i];
        const mh_graph::Node& r = g.nodes[i + 1];
        if (a.op != MH_ADD || r.op != MH_RELU || r.in[0] != a.out || m->fuse[i] || m->fuse[i + 1]) continue;
        // the ADD output is read by this RELU only, and is not a graph output or the loss
        bool only = g.loss != a.out;
        for (size_t j = 0; j < g.nodes.size() && only; ++j)
            for (int k = 0; k < g.nodes[j].nin; ++k)
                if (j != i + 1 && g.nodes[j].in[k] == a.out) only = false;
        for (int32_t o : g.outputs)
            if (o == a.out) only = false;
        if (!only) continue;
        // x + bias with x of the output shape and bias broadcast into it (never the reverse)
        const mh_shape& sx = g.syms[a.in[0]].shape;
        const mh_shape& sb = g.syms[a.in[1]].shape;
        const mh_shape& sy = g.syms[a.out].shape;
        if (!shape_eq(sx, sy) || shape_eq(sb, sy) || !broadcasts_to(sb, sy)) continue;
        m->fuse[i] = kFuseAdd;
        m->fuse[i + 1] = kFuseRelu;
    }
}

// ---------------------------------------------------------------------------------------
// programs: runs of nodes over one [R, W] view as one launch
// ---------------------------------------------------------------------------------------
// The view of a run: shape S (the largest of its first node), W its last dimension.
struct ProgView {
    mh_shape S;
    int64_t R = 0;
    int64_t W = 0;
    bool single() const { return R * W <= kProgSingle; }
    // Row instructions: a row per wavefront needs k_rows_wave's lengths, and several slabs of them
    // lose to the node's own kernels (the head over [5000, 200]: 92 us against 79).
    bool rows_ok() const { return W <= 64 || (single() && W < 2048); }
    // Gradients of a row's MAX or of a per-row operand: a row per thread, one pass over the workgroup (a
    // MAX gradient's maxima lie in LDS, kProgRows of them). Longer rows and more of them are their nodes'
    // own kernels, and the run ends there: the backward of the head over [4, 2000] 112 us in programs, 76
    // so, over [64, 128] 85 and 64, over [4000, 2] 75 and 64.
    bool row_grads_ok() const { return W <= 64 && (!single() || R <= kProgRows); }
};

static int64_t dim_from_end(const mh_shape& s, int k) { return k < s.rank ? s.dims[s.rank - 1 - k] : 1; }

// The form of shape t in the view, or -1.
static int prog_class(const ProgView& v, const mh_shape& t) {
    const int64_t n = numel(t);
    const int rank = t.rank > v.S.rank ? t.rank : v.S.rank;
    bool full = true, row = v.W > 1 && v.R > 1, col = v.R > 1 && v.W > 1;
    for (int k = 0; k < rank; ++k) {
        const int64_t a = dim_from_end(t, k), b = dim_from_end(v.S, k);
        full = full && a == b;
        row = row && a == (k == 0 ? 1 : b);
        col = col && a == (k == 0 ? b : 1);
    }
    if (full) return PC_FULL;
    if (n == 1) return PC_SCAL;
    return row ? PC_ROW : col ? PC_COL : -1;
}

// Instructions of one run and their accesses since the last barrier: an address touched under two
// thread mappings, once to write, needs a barrier between.
struct ProgBuild {
    ProgView v;
    std::vector<ProgInstr> a, b;
    std::vector<ProgSum> sums;
    int64_t part = 0;     // partial floats per workgroup
    bool cols = false;    // sums over rows
    std::unordered_map<const float*, int> reads, writes;  // address -> mapping (kAny: several)
    static constexpr int kFlat = 1, kFlatRow = 2, kRows = 3, kAny = 4;

    // The run as it was at an earlier node: the parts appended since are dropped.
    struct Mark {
        size_t na, nb, ns;
        int64_t part;
        bool cols;
    };
    Mark mark() const { return Mark{a.size(), b.size(), sums.size(), part, cols}; }
    void cut(const Mark& k) {
        a.resize(k.na);
        b.resize(k.nb);
        sums.resize(k.ns);
        part = k.part;
        cols = k.cols;
    }

    bool clash(const float* p, int map, bool write) {
        auto hit = [&](std::unordered_map<const float*, int>& m) {
            auto it = m.find(p);
            return it != m.end() && (it->second != map || map == kAny);
        };
        return p && (hit(writes) || (write && hit(reads)));
    }
    void note(std::unordered_map<const float*, int>& m, const float* p, int map) {
        if (!p) return;
        auto it = m.find(p);
        if (it == m.end()) m[p] = map;
        else if (it->second != map) it->second = kAny;
    }
    // map_of[k]: the mapping under which operands a, b, c and the output are touched
    void push(ProgInstr in, const int (&map)[4]) {
        const float* p[4] = {in.a, in.b, in.c, in.out};
        bool bar = false;
        for (int k = 0; k < 4; ++k) bar = bar || clash(p[k], map[k], k == 3);
        if (bar) {
            in.flags |= PF_BARRIER;
            reads.clear();
            writes.clear();
        }
        for (int k = 0; k < 3; ++k) note(reads, p[k], map[k]);
        note(writes, in.out, map[3]);
        a.push_back(in);
    }
    static ProgInstr instr(int op, float* out, const float* x, int cx, const float* y = nullptr, int cy = 0,
                           const float* z = nullptr, int cz = 0) {
        ProgInstr in{};
        in.op = op;
        in.out = out;
        in.a = x;
        in.b = y;
        in.c = z;
        in.cls = cx | (cy << 2) | (cz << 4);
        return in;
    }
    // elementwise over the view's elements, or its rows (co == PC_ROW)
    void ew(ProgInstr in, int co) {
        const int base = co == PC_ROW ? kFlatRow : kFlat;
        if (co == PC_ROW) in.flags |= PF_ROWDOM;
        int map[4];
        for (int k = 0; k < 3; ++k) map[k] = ((in.cls >> (2 * k)) & 3) == co ? base : kAny;
        map[3] = base;
        push(in, map);
    }
};

static bool prog_forward_node(mh_model* m, size_t i, ProgBuild& pb) {
    const mh_graph& g = m->g;
    const mh_graph::Node& nd = g.nodes[i];
    if (m->fuse[i] == kFuseRow) return false;
    int c[3] = {0, 0, 0};
    for (int k = 0; k < nd.nin; ++k)
        if ((c[k] = prog_class(pb.v, g.syms[nd.in[k]].shape)) < 0) return false;
    const int co = prog_class(pb.v, g.syms[nd.out].shape);
    const mh_shape& sx = g.syms[nd.in[0]].shape;
    float* out = m->t[nd.out];
    const float* x = m->t[nd.in[0]];
    if (is_reduce(nd.op)) {
        const int ax = axis_of(nd.attrs);
        const float div = nd.op == MH_MEAN ? (float)(ax < 0 ? numel(sx) : sx.dims[ax]) : 0.0f;
        if (ax < 0) {  // every element
            if (c[0] != PC_FULL && c[0] != PC_ROW) return false;
            if (!pb.v.single()) return false;
            ProgInstr in = ProgBuild::instr(nd.op == MH_MAX ? PO_AMAX : PO_ASUM, out, x, c[0]);
            in.f0 = div;
            if (c[0] == PC_ROW) in.flags |= PF_ROWDOM;
            const int map[4] = {ProgBuild::kAny, 0, 0, ProgBuild::kAny};
            pb.push(in, map);
            return true;
        }
        if (ax != sx.rank - 1 || c[0] != PC_FULL || co != PC_ROW || !pb.v.rows_ok()) return false;
        ProgInstr in = ProgBuild::instr(nd.op == MH_MAX ? PO_RMAX : PO_RSUM, out, x, PC_FULL);
        in.f0 = div;
        const int map[4] = {ProgBuild::kRows, 0, 0, ProgBuild::kRows};
        pb.push(in, map);
        return true;
    }
    if (co != PC_FULL && co != PC_ROW) return false;
    for (int k = 0; k < nd.nin; ++k)
        if (co == PC_ROW && c[k] != PC_ROW && c[k] != PC_SCAL) return false;
    if (is_binary(nd.op)) {
        pb.ew(ProgBuild::instr(PO_ADD + (nd.op - MH_ADD), out, x, c[0], m->t[nd.in[1]], c[1]), co);
        return true;
    }
    if (nd.nin != 1) return false;
    int op;
    switch (nd.op) {
        case MH_EXP: op = PO_EXP; break;
        case MH_LOG: op = PO_LOG; break;
        case MH_SIGMOID: op = PO_SIGMOID; break;
        case MH_RELU: op = PO_RELU; break;
        case MH_TANH: op = PO_TANH; break;
        case MH_LEAKYRELU: op = PO_LEAKY; break;
        case MH_CLIP: op = PO_CLIP; break;
        default: return false;
    }
    ProgInstr in = ProgBuild::instr(op, out, x, c[0]);
    in.f0 = op == PO_LEAKY ? nd.attrs.negative_slope : clip_lo(nd.attrs);
    in.f1 = clip_hi(nd.attrs);
    pb.ew(in, co);
    return true;
}

// Appends the node's gradient instructions; false where one of them has no program form (pb is then
// as it was).
static bool prog_backward_node(mh_model* m, size_t i, ProgBuild& pb) {
    const mh_graph& g = m->g;
    const mh_graph::Node& nd = g.nodes[i];
    if (m->fuse[i] == kFuseRow) return false;
    const float* ug = m->gr[nd.out];
    if (!ug) return true;  // no trainable operand
    int c[3] = {0, 0, 0};
    for (int k = 0; k < nd.nin; ++k)
        if ((c[k] = prog_class(pb.v, g.syms[nd.in[k]].shape)) < 0) return false;
    const int co = prog_class(pb.v, g.syms[nd.out].shape);
    const mh_shape& sx = g.syms[nd.in[0]].shape;
    const float* t1 = m->t[nd.in[0]];
    float* g1 = m->gr[nd.in[0]];
    if (is_binary(nd.op)) {
        if (co != PC_FULL && co != PC_ROW) return false;
        const float* t2 = m->t[nd.in[1]];
        float* gr[2] = {g1, m->gr[nd.in[1]]};
        // Two full gradients of several slabs: the node's own kernel reads ug once for both (a chain of
        // TANH and MUL by the input over [500, 2000], backward: 41.7 us in programs, 30.5 so).
        if (gr[0] && gr[1] && !pb.v.single() && c[0] == PC_FULL && c[1] == PC_FULL) return false;
        // Sums over the few rows of a wide slab wait on one load after another: the backward of three MUL
        // -> ADD -> RELU layers over [2, 4000] 81 us in programs, 48 with these nodes apart ([5, 1500]: 45
        // and 51).
        for (int k = 0; k < 2; ++k) {  // every part has a form, before any is appended
            if (!gr[k] || c[k] == co) continue;
            if (co != PC_FULL || c[k] == PC_SCAL) return false;
            if (c[k] == PC_ROW && !pb.v.row_grads_ok()) return false;
            if (c[k] == PC_COL) {
                if (pb.v.single() && pb.v.W > 1536) return false;
                if (pb.b.size() >= kProgMaxSums) return false;  // k_prog_final has a grid row for each
                if (!pb.v.single() && pb.v.R <= 64) return false;  // a short column's sum keeps its order
                if (gr[0] == gr[1]) return false;
                for (const ProgInstr& e : pb.b)
                    if (e.out == gr[k]) return false;
            }
        }
        for (int k = 0; k < 2; ++k) {
            if (!gr[k]) continue;
            // (kind, operands) of FBinRg: ug, then what it reads
            int kind;
            ProgInstr in;
            if (nd.op == MH_ADD || (nd.op == MH_SUB && k == 0)) {
                kind = PT_UG;
                in = ProgBuild::instr(0, gr[k], ug, co);
            } else if (nd.op == MH_SUB) {
                kind = PT_NEG;
                in = ProgBuild::instr(0, gr[k], ug, co);
            } else if (nd.op == MH_MUL) {
                kind = PT_MUL;
                in = k == 0 ? ProgBuild::instr(0, gr[k], ug, co, t2, c[1]) : ProgBuild::instr(0, gr[k], ug, co, t1, c[0]);
            } else if (k == 0) {
                kind = PT_DIV0;
                in = ProgBuild::instr(0, gr[k], ug, co, t2, c[1]);
            } else {
                kind = PT_DIV1;
                in = ProgBuild::instr(0, gr[k], ug, co, t1, c[0], t2, c[1]);
            }
            if (c[k] == co) {
                in.op = PO_G_UG + (kind - PT_UG);
                pb.ew(in, co);
            } else if (c[k] == PC_ROW) {
                in.op = PO_RUNB;
                in.slot = kind;
                int map[4];
                for (int j = 0; j < 3; ++j) {
                    const int cl = (in.cls >> (2 * j)) & 3;
                    map[j] = cl == PC_FULL || cl == PC_ROW ? ProgBuild::kRows : ProgBuild::kAny;
                }
                map[3] = ProgBuild::kRows;
                pb.push(in, map);
            } else {
                in.op = PO_CUNB;
                in.slot = kind;
                if (!pb.v.single()) {
                    in.part = pb.part;
                    pb.sums.push_back(ProgSum{gr[k], pb.part, (int32_t)pb.v.W, 0});
                    pb.part += pb.v.W;
                }
                pb.cols = true;
                pb.b.push_back(in);
            }
        }
        return true;
    }
    if (!g1) return true;
    if (is_reduce(nd.op)) {
        const int ax = axis_of(nd.attrs);
        if (ax < 0) {
            if (nd.op == MH_MAX || (c[0] != PC_FULL && c[0] != PC_ROW)) return false;
            ProgInstr in = ProgBuild::instr(PO_G_SCALE, g1, ug, PC_SCAL);
            in.f0 = nd.op == MH_SUM ? 1.0f : (float)(1.0 / (double)numel(sx));
            pb.ew(in, c[0]);
            return true;
        }
        if (ax != sx.rank - 1 || c[0] != PC_FULL || co != PC_ROW) return false;
        if (nd.op == MH_MAX) {
            if (!pb.v.row_grads_ok()) return false;
            ProgInstr in = ProgBuild::instr(PO_RMAXB, g1, t1, PC_FULL, ug, PC_ROW);
            const int map[4] = {ProgBuild::kAny, ProgBuild::kAny, 0, ProgBuild::kAny};
            pb.push(in, map);
            return true;
        }
        ProgInstr in = ProgBuild::instr(PO_G_SCALE, g1, ug, PC_ROW);
        in.f0 = nd.op == MH_SUM ? 1.0f : (float)(1.0 / (double)sx.dims[ax]);
        pb.ew(in, PC_FULL);
        return true;
    }
    if (nd.nin != 1 || (co != PC_FULL && co != PC_ROW) || c[0] != co) return false;
    int op;
    switch (nd.op) {
        case MH_EXP: op = PO_G_EXP; break;
        case MH_LOG: op = PO_G_LOG; break;
        case MH_SIGMOID: op = PO_G_SIGMOID; break;
        case MH_RELU: op = PO_G_RELU; break;
        case MH_TANH: op = PO_G_TANH; break;
        case MH_LEAKYRELU: op = PO_G_LEAKY; break;
        case MH_CLIP: op = PO_G_CLIP; break;
        default: return false;
    }
    ProgInstr in = ProgBuild::instr(op, g1, t1, c[0], ug, co);
    in.f0 = op == PO_G_LEAKY ? nd.attrs.negative_slope : clip_lo(nd.attrs);
    in.f1 = clip_hi(nd.attrs);
    pb.ew(in, co);
    return true;
}

// The view of a run that starts at node i: the largest of its operands and output.
static bool prog_view(const mh_model* m, size_t i, ProgView* v) {
    const mh_graph::Node& nd = m->g.nodes[i];
    const mh_shape* best = &m->g.syms[nd.out].shape;
    for (int k = 0; k < nd.nin; ++k)
        if (numel(m->g.syms[nd.in[k]].shape) > numel(*best)) best = &m->g.syms[nd.in[k]].shape;
    v->S = *best;
    v->W = best->dims[best->rank - 1];
    const int64_t n = numel(*best);
    if (n < 2 || v->W < 2 || n >= ((int64_t)1 << 31)) return false;
    v->R = n / v->W;
    return true;
}

// Rows of a slab, and whether the run is worth a program: slabs of about 2048 elements, of at least
// 8 rows where sums over rows leave a partial per slab. Measured, a training step of MUL -> ADD ->
// RELU layers, nodes one by one against programs: 24 layers of [32, 32] 530-630 and 165 us, 3 of
// [1902, 31] 151 and 75, 3 of [3000, 300] 146 and 106. Wider slabs go node by node (8 rows of 1000: 96
// and 124), and so do views of more than a million elements, where the kernels stream at memory speed
// and one workgroup a slab does not: 8 TANH in a row over [16384, 500] 366 us node by node and 472 as
// programs, over [60000, 20] 89 and 111, 4 layers of [16384, 500] 613 and 658, the head over [2^20, 10]
// 394 and 480. One kind there would gain and is left: narrow layers, for their sums over rows (4 of
// [20000, 64] 204 and 115).
static bool prog_shape(const ProgBuild& pb, ProgRun* r) {
    const int64_t R = pb.v.R, W = pb.v.W;
    if (pb.v.single()) {
        r->rpw = (int32_t)R;
        r->nwg = 1;
        return pb.cols || pb.a.size() >= 2;
    }
    int64_t rpw = (2048 + W - 1) / W;
    if (pb.cols && rpw < 8) rpw = 8;
    if (rpw > kProgRows) rpw = kProgRows;
    const int64_t nwg = (R + rpw - 1) / rpw;
    if (nwg < 2 || rpw * W > 4096 || R * W > kProgMax) return false;
    r->rpw = (int32_t)rpw;
    r->nwg = (int32_t)nwg;
    // two launches cost less than a program's two instructions one after another (SUB -> EXP over [200,
    // 2000], 11 us in one, 5.6 in two)
    return pb.cols || pb.a.size() >= 4;
}

struct ProgPlan {
    std::vector<ProgInstr> instrs;
    std::vector<ProgSum> sums;
    size_t part = 0;
    std::vector<std::pair<size_t, size_t>> at;  // per segment: first instruction, first sum
};

static void prog_keep(ProgBuild& pb, int first, int last, ProgPlan& plan, std::vector<mh_model::Segment>& segs,
                      std::vector<int>& of) {
    mh_model::Segment sg;
    sg.first = first;
    sg.last = last;
    ProgRun& r = sg.run;
    // a single node only for its sums over rows: wherever a view has a program these go through it,
    // so that their order does not depend on what the node's neighbours are
    if ((last == first && !pb.cols) || !prog_shape(pb, &r)) return;
    r.R = pb.v.R;
    r.W = (int32_t)pb.v.W;
    r.na = (int)pb.a.size();
    r.nb = (int)pb.b.size();
    r.nsums = (int)pb.sums.size();
    for (ProgInstr& in : pb.a) in.part *= r.nwg;
    for (ProgInstr& in : pb.b) in.part *= r.nwg;
    for (ProgSum& u : pb.sums) {
        u.part *= r.nwg;
        if (u.ncol > r.maxcol) r.maxcol = u.ncol;
    }
    const size_t part = (size_t)pb.part * (size_t)r.nwg;
    if (part > plan.part) plan.part = part;
    plan.at.emplace_back(plan.instrs.size(), plan.sums.size());
    plan.instrs.insert(plan.instrs.end(), pb.a.begin(), pb.a.end());
    plan.instrs.insert(plan.instrs.end(), pb.b.begin(), pb.b.end());
    plan.sums.insert(plan.sums.end(), pb.sums.begin(), pb.sums.end());
    for (int j = first; j <= last; ++j) of[j] = (int)segs.size();
    segs.push_back(sg);
}

// A fused bias + RELU pair is not split between a program and its kernels.
static bool prog_cut_ok(const mh_model* m, int first, int last) {
    const int nn = (int)m->g.nodes.size();
    return m->fuse[first] != kFuseRelu && !(last + 1 < nn && m->fuse[last] == kFuseAdd);
}

static void plan_programs(mh_model* m, ProgPlan& plan) {
    const int nn = (int)m->g.nodes.size();
    m->fseg_of.assign(nn, -1);
    m->bseg_of.assign(nn, -1);
    for (int i = 0; i < nn;) {
        ProgBuild pb;
        ProgBuild::Mark ok{};  // the longest run so far that may end there
        int last = -1;
        if (prog_view(m, i, &pb.v) && m->fuse[i] != kFuseRelu) {
            for (int j = i; j < nn; ++j) {
                if (!prog_forward_node(m, j, pb)) break;
                if (prog_cut_ok(m, i, j)) {
                    ok = pb.mark();
                    last = j;
                }
            }
        }
        if (last >= 0) {
            pb.cut(ok);
            prog_keep(pb, i, last, plan, m->fseg, m->fseg_of);
        }
        i = last >= i ? last + 1 : i + 1;
    }
    if (m->grad_floats == 0) return;
    for (int i = nn - 1; i >= 0;) {
        ProgBuild pb;
        ProgBuild::Mark ok{};
        int first = nn;
        if (prog_view(m, i, &pb.v) && m->fuse[i] != kFuseAdd) {
            for (int j = i; j >= 0; --j) {
                if (!prog_backward_node(m, j, pb)) break;
                if (prog_cut_ok(m, j, i)) {
                    ok = pb.mark();
                    first = j;
                }
            }
        }
        if (first <= i) {
            pb.cut(ok);
            prog_keep(pb, first, i, plan, m->bseg, m->bseg_of);
        }
        i = first <= i ? first - 1 : i - 1;
    }
}

static size_t pad256(size_t b) { return (b + 255) & ~(size_t)255; }

// Plans the model's programs and places them on the device.
static int build_programs(mh_model* m) {
    ProgPlan plan;
    plan_programs(m, plan);
    if (plan.at.empty()) return MH_OK;
    const size_t ib = pad256(plan.instrs.size() * sizeof(ProgInstr)), sb = pad256(plan.sums.size() * sizeof(ProgSum));
    MH_TRY(mh_malloc(&m->prog_mem, ib + sb));
    if (plan.part) MH_TRY(mh_malloc(reinterpret_cast<void**>(&m->prog_part), plan.part * sizeof(float)));
    MH_TRY(mh_memcpy_h2d(m->prog_mem, plan.instrs.data(), plan.instrs.size() * sizeof(ProgInstr)));
    char* sums = static_cast<char*>(m->prog_mem) + ib;
    MH_TRY(mh_memcpy_h2d(sums, plan.sums.data(), plan.sums.size() * sizeof(ProgSum)));
    size_t k = 0;
    for (auto* segs : {&m->fseg, &m->bseg})
        for (mh_model::Segment& s : *segs) {
            s.run.prog = static_cast<const ProgInstr*>(m->prog_mem) + plan.at[k].first;
            s.run.sums = reinterpret_cast<const ProgSum*>(sums) + plan.at[k].second;
            s.run.part = m->prog_part;
            ++k;
        }
    return MH_OK;
}

static int run_forward_node(mh_model* m, size_t i) {
    const mh_graph& g = m->g;
    const mh_graph::Node& nd = g.nodes[i];
    float* res = m->t[nd.out];
    const mh_shape& so = g.syms[nd.out].shape;
    const float* a = m->t[nd.in[0]];
    const mh_shape& sa = g.syms[nd.in[0]].shape;
    const int64_t n = numel(so);
    if (m->fuse[i] == kFuseRow) {  // a row group runs as one kernel at its first node
        const mh_model::RowGroup& r = m->rows[m->row_of[i]];
        if ((int)i != r.first) return MH_OK;
        switch (r.graph) {
            case 0: return mh_softmax_log_mul_mean_fwd(m->t[r.out], m->t[r.x], m->t[r.target], r.rows, r.K);
            case 1: return cross_entropy_fwd_c(m->t[r.out], m->t[r.x], m->t[r.target], r.rows, r.K, r.scale);
            case 2: return mh_softmax_fwd(m->t[r.out], m->t[r.x], r.rows, r.K);
            default: return mh_logsoftmax_fwd(m->t[r.out], m->t[r.x], r.rows, r.K);
        }
    }
    if (m->fuse[i] == kFuseAdd) {  // ADD + the RELU after it: writes both outputs
        const mh_graph::Node& r = g.nodes[i + 1];
        return mh_bias_relu_fwd(res, m->t[r.out], a, &sa, m->t[nd.in[1]], &g.syms[nd.in[1]].shape);
    }
    if (m->fuse[i] == kFuseRelu) return MH_OK;
    if (is_binary(nd.op)) return mh_binary_fwd(nd.op, res, &so, a, &sa, m->t[nd.in[1]], &g.syms[nd.in[1]].shape);
    if (nd.op == MH_POW) return mh_pow_fwd(res, a, n, m->t[nd.in[1]]);
    if (is_unary(nd.op)) return mh_unary_fwd(nd.op, res, a, n);
    if (is_reduce(nd.op)) return mh_reduce_fwd(nd.op, res, a, &sa, axis_of(nd.attrs));
    if (nd.op == MH_FMA) return mh_fma_fwd(res, a, m->t[nd.in[1]], m->t[nd.in[2]], n);
    if (nd.op == MH_LEAKYRELU) return mh_leakyrelu_fwd(res, a, n, nd.attrs.negative_slope);
    return mh_clip_fwd(res, a, n, clip_lo(nd.attrs), clip_hi(nd.attrs));
}

// Model.backward's per-node step (model.mojo:214-330): backward_op for every trainable
// operand, in operand order, each accumulating into that operand's gradient.
static int run_backward_node(mh_model* m, size_t i) {
    const mh_graph& g = m->g;
    const mh_graph::Node& nd = g.nodes[i];
    const float* ug = m->gr[nd.out];
    if (!ug) return MH_OK;  // no trainable operand
    const mh_shape& so = g.syms[nd.out].shape;
    const int32_t* in = nd.in;
    if (m->fuse[i] == kFuseRow) {  // a row group's backward runs at its last node
        const mh_model::RowGroup& r = m->rows[m->row_of[i]];
        if ((int)i != r.last) return MH_OK;
        float* gx = m->gr[r.x];
        switch (r.graph) {
            case 0: return mh_softmax_log_mul_mean_bwd_accum(gx, m->t[r.x], m->t[r.target], ug, r.rows, r.K);
            case 1: return cross_entropy_bwd_c(gx, m->t[r.x], m->t[r.target], ug, r.rows, r.K, r.scale);
            case 2: return mh_softmax_bwd_accum(gx, m->t[r.x], ug, r.rows, r.K);
            default: return mh_logsoftmax_bwd_accum(gx, m->t[r.x], ug, r.rows, r.K);
        }
    }
    if (m->fuse[i] == kFuseRelu) {  // RELU, then the ADD before it
        const mh_graph::Node& a = g.nodes[i - 1];
        float* gy = m->gr[a.out];
        float* gx = m->gr[a.in[0]];
        float* gb = m->gr[a.in[1]];
        return mh_bias_relu_bwd_accum(gy, gx, gb, m->t[a.out], ug, &so, &g.syms[a.in[1]].shape);
    }
    if (m->fuse[i] == kFuseAdd) return MH_OK;
    const float* t1 = m->t[in[0]];
    const mh_shape& s1 = g.syms[in[0]].shape;
    const int64_t n1 = numel(s1);
    if (is_binary(nd.op)) {
        const float* t2 = m->t[in[1]];
        const mh_shape& s2 = g.syms[in[1]].shape;
        float* g1 = m->gr[in[0]];
        float* g2 = m->gr[in[1]];
        // same result, one pass (also for one symbol used twice: one gradient, id 0's part first)
        if (g1 && g2 && shape_eq(s1, s2) && shape_eq(s1, so))
            return mh_binary_bwd_accum2(nd.op, g1, g2, ug, t1, t2, &s1);
        if (g1) MH_TRY(mh_binary_bwd_accum(nd.op, 0, g1, &s1, ug, &so, t1, &s1, t2, &s2));
        if (g2) MH_TRY(mh_binary_bwd_accum(nd.op, 1, g2, &s2, ug, &so, t1, &s1, t2, &s2));
        return MH_OK;
    }
    if (nd.op == MH_POW)  // both operand gradients in one pass where both are trainable
        return mh_pow_bwd_accum2(m->gr[in[0]], m->gr[in[1]], t1, m->t[in[1]], ug, n1);
    if (nd.op == MH_FMA) {
        for (int j = 0; j < 3; ++j)
            if (m->gr[in[j]]) MH_TRY(mh_fma_bwd_accum(j, m->gr[in[j]], ug, t1, m->t[in[1]], n1));
        return MH_OK;
    }
    float* g1 = m->gr[in[0]];
    if (!g1) return MH_OK;
    if (is_unary(nd.op)) return mh_unary_bwd_accum(nd.op, g1, t1, ug, n1);
    if (is_reduce(nd.op)) return mh_reduce_bwd_accum(nd.op, g1, t1, &s1, ug, axis_of(nd.attrs));
    if (nd.op == MH_LEAKYRELU) return mh_leakyrelu_bwd_accum(g1, t1, ug, n1, nd.attrs.negative_slope);
    return mh_clip_bwd_accum(g1, t1, ug, n1, clip_lo(nd.attrs), clip_hi(nd.attrs));
}

// Nodes [0, nodes) forward, and every node backward: programs where they cover a run, else a node
// at a time.
static int run_forward(mh_model* m, int32_t nodes) {
    for (int32_t i = 0; i < nodes; ++i) {
        const int sg = m->fseg_of[i];
        if (sg >= 0 && m->fseg[sg].first == i && m->fseg[sg].last < nodes) {
            MH_TRY(prog_launch(m->fseg[sg].run));
            i = m->fseg[sg].last;
        } else {
            MH_TRY(run_forward_node(m, (size_t)i));
        }
    }
    return MH_OK;
}

static int run_backward(mh_model* m) {
    for (int32_t i = (int32_t)m->g.nodes.size() - 1; i >= 0; --i) {
        const int sg = m->bseg_of[i];
        if (sg >= 0 && m->bseg[sg].last == i) {
            MH_TRY(prog_launch(m->bseg[sg].run));
            i = m->bseg[sg].first;
        } else {
            MH_TRY(run_backward_node(m, (size_t)i));
        }
    }
    return MH_OK;
}

static int write_inputs(mh_model* m, int32_t ninputs, const float* const* inputs, int where) {
    const mh_graph& g = m->g;
    if (ninputs != (int32_t)g.inputs.size())
        return fail(MH_ERR_INVALID, "%d inputs given, the graph has %zu", ninputs, g.inputs.size());
    if (ninputs > 0 && !inputs) return fail(MH_ERR_NULL, "null input table");
    if (where != MH_FROM_HOST && where != MH_FROM_DEVICE) return fail(MH_ERR_INVALID, "bad input location %d", where);
    for (int32_t k = 0; k < ninputs; ++k) {
        const int32_t s = g.inputs[k];
        MH_TRY(copy_in(m->t[s], inputs[k], (size_t)numel(g.syms[s].shape), where));
    }
    if (where == MH_FROM_HOST && ninputs > 0) MH_HIP(hipStreamSynchronize(ctx().stream));  // pageable sources
    return MH_OK;
}

// The ops of one pass, enqueued on the library stream (no synchronisation): forward = every
// node; backward = the loss gradient seeded with 1.0, then every node in reverse.
static int check_pass(const mh_model* m, int pass) {
    if (pass == MH_PASS_FORWARD) return MH_OK;
    if (pass != MH_PASS_BACKWARD && pass != MH_PASS_STEP) return fail(MH_ERR_INVALID, "unknown pass %d", pass);
    if (m->g.loss < 0) return fail(MH_ERR_INVALID, "backward pass: the graph has no loss symbol");
    if (!m->gr[m->g.loss]) return fail(MH_ERR_INVALID, "backward pass: the loss is not trainable");
    return MH_OK;
}

static int enqueue_pass(mh_model* m, int pass) {
    const mh_graph& g = m->g;
    if (pass == MH_PASS_STEP && m->grad_arena)  // parameters.grads.set_zero (collection.mojo:221-224)
        MH_TRY(mh_zero(m->grad_arena, (int64_t)m->grad_floats));
    if (pass == MH_PASS_FORWARD || pass == MH_PASS_STEP)
        MH_TRY(run_forward(m, (int32_t)g.nodes.size()));
    if (pass == MH_PASS_FORWARD) return MH_OK;
    MH_TRY(mh_fill(m->gr[g.loss], 1.0f, numel(g.syms[g.loss].shape)));  // model.mojo:176-180
    return run_backward(m);
}

static void drop_graphs(mh_model* m) {
    for (int p = 0; p < 3; ++p) {
        if (m->graph[p]) {
            (void)hipGraphExecDestroy(m->graph[p]);
            (void)graph_release(m->graph_epoch[p]);
        }
        m->graph[p] = nullptr;
    }
}

static int execute(mh_model* m, int32_t nodes, const char* what) {
    PassScope ps;
    MH_TRY(run_forward(m, nodes));
    return ps.end(what);
}

}  // namespace mh

using namespace mh;

extern "C" {

// ---------------------------------------------------------------------------------------
// Graph (graph.mojo:33-217)
// ---------------------------------------------------------------------------------------
int mh_graph_create(mh_graph** out) {
    if (!out) return fail(MH_ERR_NULL, "mh_graph_create: null out");
    *out = new (std::nothrow) mh_graph();
    if (!*out) return fail(MH_ERR_INVALID, "mh_graph_create: out of host memory");
    return MH_OK;
}

int mh_graph_destroy(mh_graph* g) {
    delete g;
    return MH_OK;
}

int mh_graph_input(mh_graph* g, const mh_shape* pshape, int trainable, int32_t* sym) {
    if (!g || !sym) return fail(MH_ERR_NULL, "mh_graph_input: null argument");
    MH_SHAPE_ARG(shape);
    MH_TRY(add_symbol(g, shape, trainable, MH_SYM_INPUT, sym));
    g->inputs.push_back(*sym);
    return MH_OK;
}

int mh_graph_param(mh_graph* g, const mh_shape* pshape, int trainable, const float* data, int64_t ndata,
                   int32_t* sym) {
    if (!g || !sym) return fail(MH_ERR_NULL, "mh_graph_param: null argument");
    MH_SHAPE_ARG(shape);
    MH_TRY(check_shape(shape, "param"));
    if (ndata < 0 || (ndata > 0 && !data)) return fail(MH_ERR_INVALID, "mh_graph_param: bad init data");
    if (ndata > 0 && ndata != numel(shape))
        return fail(MH_ERR_SHAPE, "mh_graph_param: %lld init values for %lld elements", (long long)ndata,
                    (long long)numel(shape));
    MH_TRY(add_symbol(g, shape, trainable, MH_SYM_PARAM, sym));
    if (ndata > 0) {
        g->syms.back().init_off = (int64_t)g->init_data.size();
        g->init_data.insert(g->init_data.end(), data, data + ndata);
    }
    g->params.push_back(*sym);
    return MH_OK;
}

int mh_graph_scalar(mh_graph* g, float value, int32_t* sym) {
    const mh_shape s = flat_shape(1);
    return mh_graph_param(g, &s, 0, &value, 1, sym);
}

int mh_graph_op(mh_graph* g, int op, int32_t noperands, const int32_t* operands, const mh_attrs* attrs,
                int32_t* sym) {
    if (!g || !sym || (noperands > 0 && !operands)) return fail(MH_ERR_NULL, "mh_graph_op: null argument");
    const int ar = op_arity(op);
    if (ar == 0) return fail(MH_ERR_OP, "mh_graph_op: operator %d is not on this path", op);
    if (noperands != ar) return fail(MH_ERR_INVALID, "mh_graph_op: operator %d takes %d operands, got %d", op, ar, noperands);
    for (int k = 0; k < ar; ++k) MH_TRY(check_sym(g, operands[k]));
    mh_attrs at{};
    if (attrs) at = *attrs;
    mh_shape rs;
    MH_TRY(result_shape(*g, op, ar, operands, at, &rs));
    int tr = 0;  // result_trainable (graph.mojo:212-217)
    for (int k = 0; k < ar; ++k) tr |= g->syms[operands[k]].trainable;
    MH_TRY(add_symbol(g, rs, tr, MH_SYM_NODE, sym));
    mh_graph::Node nd;
    nd.op = op;
    nd.nin = ar;
    for (int k = 0; k < 3; ++k) nd.in[k] = k < ar ? operands[k] : -1;
    nd.out = *sym;
    nd.attrs = at;
    g->nodes.push_back(nd);
    return MH_OK;
}

int mh_graph_out(mh_graph* g, int32_t sym) {
    if (!g) return fail(MH_ERR_NULL, "mh_graph_out: null graph");
    MH_TRY(check_sym(g, sym));
    g->outputs.push_back(sym);
    return MH_OK;
}

int mh_graph_loss(mh_graph* g, int32_t sym) {
    if (!g) return fail(MH_ERR_NULL, "mh_graph_loss: null graph");
    MH_TRY(check_sym(g, sym));
    g->loss = sym;
    return MH_OK;
}

int mh_graph_symbol(const mh_graph* g, int32_t sym, mh_shape* shape, int* trainable, int* kind) {
    if (!g) return fail(MH_ERR_NULL, "mh_graph_symbol: null graph");
    MH_TRY(check_sym(g, sym));
    if (shape) *shape = g->syms[sym].shape;
    if (trainable) *trainable = g->syms[sym].trainable;
    if (kind) *kind = g->syms[sym].kind;
    return MH_OK;
}

int mh_graph_counts(const mh_graph* g, int32_t* nsymbols, int32_t* nnodes, int32_t* ninputs, int32_t* nparams,
                    int32_t* noutputs) {
    if (!g) return fail(MH_ERR_NULL, "mh_graph_counts: null graph");
    if (nsymbols) *nsymbols = (int32_t)g->syms.size();
    if (nnodes) *nnodes = (int32_t)g->nodes.size();
    if (ninputs) *ninputs = (int32_t)g->inputs.size();
    if (nparams) *nparams = (int32_t)g->params.size();
    if (noutputs) *noutputs = (int32_t)g->outputs.size();
    return MH_OK;
}

// ---------------------------------------------------------------------------------------
// Model (model.mojo:55-340)
// ---------------------------------------------------------------------------------------
int mh_model_create(const mh_graph* g, uint64_t flags, mh_model** out) {
    if (!g || !out) return fail(MH_ERR_NULL, "mh_model_create: null argument");
    *out = nullptr;
    MH_TRY(require_init());
    mh_model* m = new (std::nothrow) mh_model();
    if (!m) return fail(MH_ERR_INVALID, "mh_model_create: out of host memory");
    m->g = *g;
    m->flags = flags;
    const size_t ns = g->syms.size();
    std::vector<size_t> toff(ns), goff(ns, (size_t)-1);
    // allocate_tensor_memory / allocate_grad_memory. The trainable parameters come first in
    // both arenas, in the same order with the same slot sizes, so that parameters and their
    // gradients form two parallel spans an optimizer updates in one launch; then every other
    // symbol in creation order.
    auto is_tparam = [&](size_t s) { return g->syms[s].kind == MH_SYM_PARAM && g->syms[s].trainable; };
    for (int pass = 0; pass < 2; ++pass) {
        for (size_t s = 0; s < ns; ++s) {
            if (is_tparam(s) != (pass == 0)) continue;
            toff[s] = m->arena_floats;
            m->arena_floats += slot_floats(g->syms[s].shape);
            if (g->syms[s].trainable) {
                goff[s] = m->grad_floats;
                m->grad_floats += slot_floats(g->syms[s].shape);
            }
        }
        if (pass == 0) m->param_span = m->arena_floats;
    }
    int rc = MH_OK;
    if (m->arena_floats) rc = mh_malloc(reinterpret_cast<void**>(&m->arena), m->arena_floats * sizeof(float));
    if (rc == MH_OK && m->grad_floats)
        rc = mh_malloc(reinterpret_cast<void**>(&m->grad_arena), m->grad_floats * sizeof(float));
    if (rc == MH_OK) {
        m->t.resize(ns);
        m->gr.assign(ns, nullptr);
        for (size_t s = 0; s < ns; ++s) {
            m->t[s] = m->arena + toff[s];
            if (goff[s] != (size_t)-1) m->gr[s] = m->grad_arena + goff[s];
        }
        // Tensor[f32](shape) is zero-initialised (tensor.mojo:266); parameters with data
        // get it copied in (model.mojo:353-370)
        PassScope ps;
        if (m->arena) rc = mh_zero(m->arena, (int64_t)m->arena_floats);
        if (rc == MH_OK && m->grad_arena) rc = mh_zero(m->grad_arena, (int64_t)m->grad_floats);
        for (size_t s = 0; s < ns && rc == MH_OK; ++s) {
            const mh_graph::Sym& y = g->syms[s];
            if (y.kind == MH_SYM_PARAM && y.init_off >= 0)
                rc = copy_in(m->t[s], g->init_data.data() + y.init_off, (size_t)numel(y.shape), MH_FROM_HOST);
        }
        // the host init data is pageable: wait for its copies whatever the caller's flags
        if (rc == MH_OK) rc = hip_check(hipStreamSynchronize(ctx().stream), "mh_model_create");
        (void)ps;
    }
    if (rc == MH_OK) {
        m->n_inference = inference_nodes(m->g);
        plan_fusion(m);
        rc = build_programs(m);
    }
    if (rc != MH_OK) {
        if (m->arena) mh_free(m->arena);
        if (m->grad_arena) mh_free(m->grad_arena);
        if (m->prog_mem) mh_free(m->prog_mem);
        if (m->prog_part) mh_free(m->prog_part);
        delete m;
        return rc;
    }
    *out = m;
    return MH_OK;
}

int mh_model_destroy(mh_model* m) {
    if (!m) return MH_OK;
    drop_graphs(m);
    int rc = MH_OK;
    if (m->arena) rc = mh_free(m->arena);
    if (m->grad_arena) {
        const int r2 = mh_free(m->grad_arena);
        if (rc == MH_OK) rc = r2;
    }
    for (void* p : {m->prog_mem, static_cast<void*>(m->prog_part)})
        if (p) {
            const int r2 = mh_free(p);
            if (rc == MH_OK) rc = r2;
        }
    delete m;
    return rc;
}

int mh_model_forward(mh_model* m, int32_t ninputs, const float* const* inputs, int where) {
    MH_TRACE("mh_model_forward");
    if (!m) return fail(MH_ERR_NULL, "mh_model_forward: null model");
    MH_TRY(require_init());
    MH_TRY(write_inputs(m, ninputs, inputs, where));
    return execute(m, (int32_t)m->g.nodes.size(), "mh_model_forward");
}

int mh_model_inference(mh_model* m, int32_t ninputs, const float* const* inputs, int where) {
    MH_TRACE("mh_model_inference");
    if (!m) return fail(MH_ERR_NULL, "mh_model_inference: null model");
    if (m->n_inference < 0) return fail(MH_ERR_INVALID, "mh_model_inference: the graph has no output");
    MH_TRY(require_init());
    MH_TRY(write_inputs(m, ninputs, inputs, where));
    int32_t nodes = m->n_inference;
    // a fused ADD + RELU pair is never split by the inference cut
    if (nodes > 0 && nodes < (int32_t)m->fuse.size() && m->fuse[nodes - 1] == kFuseAdd) ++nodes;
    if (nodes > 0 && nodes < (int32_t)m->fuse.size() && m->fuse[nodes - 1] == kFuseRow)
        nodes = m->rows[m->row_of[nodes - 1]].last + 1;  // never cut a row group
    return execute(m, nodes, "mh_model_inference");
}

int mh_model_backward(mh_model* m, int32_t nupper, const float* const* upper_grads, int where) {
    MH_TRACE("mh_model_backward");
    if (!m) return fail(MH_ERR_NULL, "mh_model_backward: null model");
    MH_TRY(require_init());
    const mh_graph& g = m->g;
    if (g.nodes.empty()) return MH_OK;
    PassScope ps;
    if (nupper == 0) {  // model.mojo:176-180: seed the loss gradient with 1.0
        if (g.loss < 0) return fail(MH_ERR_INVALID, "mh_model_backward: no loss symbol and no upper grads");
        if (!m->gr[g.loss]) return fail(MH_ERR_INVALID, "mh_model_backward: the loss is not trainable");
        MH_TRY(mh_fill(m->gr[g.loss], 1.0f, numel(g.syms[g.loss].shape)));
    } else {  // model.mojo:181-193: the last node's output gradient is a copy of the given one
        if (!upper_grads) return fail(MH_ERR_NULL, "mh_model_backward: null upper grads");
        if (where != MH_FROM_HOST && where != MH_FROM_DEVICE)
            return fail(MH_ERR_INVALID, "bad upper-grad location %d", where);
        const int32_t last = g.nodes.back().out;
        if (!m->gr[last]) return fail(MH_ERR_INVALID, "mh_model_backward: the last node output is not trainable");
        MH_TRY(copy_in(m->gr[last], upper_grads[0], (size_t)numel(g.syms[last].shape), where));
    }
    MH_TRY(run_backward(m));
    if (nupper != 0 && where == MH_FROM_HOST) {  // pageable source: wait whatever the flags
        MH_HIP(hipStreamSynchronize(ctx().stream));
    }
    return ps.end("mh_model_backward");
}

int mh_model_capture(mh_model* m, int pass) {
    MH_TRACE("mh_model_capture");
    if (!m) return fail(MH_ERR_NULL, "mh_model_capture: null model");
    MH_TRY(require_init());
    MH_TRY(check_pass(m, pass));
    hipStream_t st = ctx().stream;
    {  // run the pass once: library buffers reach the sizes the pass needs before capture
        PassScope ps;
        MH_TRY(enqueue_pass(m, pass));
        MH_HIP(hipStreamSynchronize(st));
    }
    PassScope ps;
    MH_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    const int rc = enqueue_pass(m, pass);
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(st, &graph);
    if (rc != MH_OK || e != hipSuccess) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc != MH_OK ? rc : hip_check(e, "mh_model_capture: hipStreamEndCapture");
    }
    hipGraphExec_t exec = nullptr;
    const hipError_t e2 = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    MH_HIP(e2);
    if (m->graph[pass]) {
        (void)hipGraphExecDestroy(m->graph[pass]);
        (void)graph_release(m->graph_epoch[pass]);
    }
    graph_retain();
    m->graph[pass] = exec;
    m->graph_epoch[pass] = ctx().epoch;
    return MH_OK;
}

int mh_model_replay(mh_model* m, int pass) {
    MH_TRACE("mh_model_replay");
    if (!m) return fail(MH_ERR_NULL, "mh_model_replay: null model");
    MH_TRY(require_init());
    if (pass != MH_PASS_FORWARD && pass != MH_PASS_BACKWARD && pass != MH_PASS_STEP)
        return fail(MH_ERR_INVALID, "unknown pass %d", pass);
    if (!m->graph[pass]) return fail(MH_ERR_INVALID, "mh_model_replay: pass %d has not been captured", pass);
    if (m->graph_epoch[pass] != ctx().epoch)
        return fail(MH_ERR_INVALID, "mh_model_replay: pass %d was captured before the last mh_shutdown; capture it again",
                    pass);
    MH_HIP(hipGraphLaunch(m->graph[pass], ctx().stream));
    return finish("mh_model_replay");
}

int mh_model_tensor(mh_model* m, int32_t sym, float** dptr) {
    if (!m || !dptr) return fail(MH_ERR_NULL, "mh_model_tensor: null argument");
    MH_TRY(check_sym(&m->g, sym));
    *dptr = m->t[sym];
    return MH_OK;
}

int mh_model_grad(mh_model* m, int32_t sym, float** dptr) {
    if (!m || !dptr) return fail(MH_ERR_NULL, "mh_model_grad: null argument");
    MH_TRY(check_sym(&m->g, sym));
    if (!m->gr[sym]) return fail(MH_ERR_INVALID, "mh_model_grad: symbol %d is not trainable", sym);
    *dptr = m->gr[sym];
    return MH_OK;
}

int mh_model_zero_grad(mh_model* m) {
    MH_TRACE("mh_model_zero_grad");
    if (!m) return fail(MH_ERR_NULL, "mh_model_zero_grad: null model");
    if (!m->grad_arena) return MH_OK;
    return mh_zero(m->grad_arena, (int64_t)m->grad_floats);
}

int mh_model_param_span(mh_model* m, float** params, float** grads, int64_t* n) {
    if (!m || !params || !grads || !n) return fail(MH_ERR_NULL, "mh_model_param_span: null argument");
    *params = m->param_span ? m->arena : nullptr;
    *grads = m->param_span ? m->grad_arena : nullptr;
    *n = (int64_t)m->param_span;
    return MH_OK;
}

int mh_model_info(const mh_model* m, int32_t* n_inference_nodes, int64_t* tensor_bytes, int64_t* grad_bytes,
                  int32_t* fused_groups) {
    if (!m) return fail(MH_ERR_NULL, "mh_model_info: null model");
    if (n_inference_nodes) *n_inference_nodes = m->n_inference;
    if (tensor_bytes) *tensor_bytes = (int64_t)(m->arena_floats * sizeof(float));
    if (grad_bytes) *grad_bytes = (int64_t)(m->grad_floats * sizeof(float));
    if (fused_groups) {
        int32_t c = 0;
        for (int f : m->fuse) c += f == kFuseAdd;
        c += (int32_t)m->rows.size();
        *fused_groups = c;
    }
    return MH_OK;
}

}  // extern "C"
