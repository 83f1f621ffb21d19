// mh_program.hip -- runs of a model's nodes as one launch (the executor's programs).
//
// A node of a model is one or two launches of 2-4 us at small sizes, whatever its work: a training
// step of 24 MUL -> ADD -> RELU layers over [32, 32] was 195 launches, 540 us for 20 KB of tensors.
// Over larger tensors each launch reads back from memory what the one before it wrote. A run of
// consecutive nodes over one [R, W] view (every tensor full [R, W], per row [R, 1], per column
// [1, W] or one element) therefore runs as a program: an instruction list in device memory that
// each workgroup walks over its own slab of whole rows, every instruction reading and writing the
// model's slots exactly as the node's own kernel does, so that a value is re-read from the caches
// its workgroup just wrote it through. Only the sums over rows (the gradients of per-column
// operands) cross slabs.
//
// One slab (up to kProgSingle elements): a workgroup of 1024 threads finishes those sums itself,
// and reduces over all elements, in the order the single kernels use. Several slabs: workgroups of
// 256 threads leave partials, one short launch adds them in slab order (k_prog_final).
//
// Thread mappings: elementwise instructions take the slab's quads in flat order, so a chain of them
// needs no barrier (each thread reads what it wrote); row instructions take a row per thread (W <=
// 64, element order) or per wavefront (W < 2048, k_rows_wave's order). The planner marks the
// instructions that need a barrier before them, and moves the sums over rows behind the rest,
// where every one is independent: a wavefront each.
#include <cfloat>

#include "mh_functors.h"
#include "mh_program.h"

namespace mh {

// Cached accesses, unlike the single kernels' streams: what an instruction writes the next ones read
// (streamed, the 3 layers of [7805, 77] took 134 us instead of 114).
__device__ __forceinline__ float ld_c(const float* p) { return *p; }
__device__ __forceinline__ void st_c(float* p, float v) { *p = v; }
__device__ __forceinline__ vf4 ld_c4(const float* p) { return *reinterpret_cast<const vf4u*>(p); }
__device__ __forceinline__ void st_c4(float* p, vf4 v) { *reinterpret_cast<vf4u*>(p) = v; }

// ---------------------------------------------------------------------------------------
// operands
// ---------------------------------------------------------------------------------------
struct Slab {
    int64_t e0;    // first element
    int64_t r0;    // first row
    int32_t rows;  // rows of this slab
    int32_t W;     // columns
    FastDiv fw;
};

// One element of an operand: element e of the view, at row r and column c.
__device__ __forceinline__ float prog_val(const float* p, int cls, int64_t e, int64_t r, int32_t c) {
    return cls == PC_FULL ? ld_c(p + e) : p[cls == PC_ROW ? r : cls == PC_COL ? c : 0];
}

// A thread's quad of the slab: its first element le and each element's row of the slab and column,
// found once and used by every instruction (an instruction of a small program is a chain of
// dependent operations on one wavefront per SIMD: its count of them is its time).
struct Pos {
    uint32_t le;
    uint32_t r[4], c[4];
    int n;  // live elements, 0 to 4
};
__device__ __forceinline__ Pos prog_pos(const Slab& s, int32_t le) {
    Pos p;
    const int32_t cnt = s.rows * s.W;
    p.n = le >= cnt ? 0 : (cnt - le < 4 ? cnt - le : 4);
    p.le = (uint32_t)le;
    uint32_t r = fdiv((uint32_t)le, s.fw), c = (uint32_t)le - r * (uint32_t)s.W;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        p.r[j] = r;
        p.c[j] = c;
        if (++c == (uint32_t)s.W) {
            c = 0;
            ++r;
        }
    }
    return p;
}

// A uniform base and a 32-bit offset in floats: one load with no address arithmetic.
__device__ __forceinline__ const float* prog_at(const float* p, uint32_t i) {
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + (uint32_t)(4u * i));
}

// Elements of a live quad (n == 4). whole: W % 4 == 0, a quad lies in one row.
__device__ __forceinline__ vf4 prog_quad(const float* p, int cls, int64_t e0, int64_t r0, const Pos& q, bool whole) {
    if (cls == PC_FULL) return ld_c4(prog_at(p + e0, q.le));
    if (cls == PC_COL && whole) return ld_c4(prog_at(p, q.c[0]));
    if (cls == PC_COL) return vf4{*prog_at(p, q.c[0]), *prog_at(p, q.c[1]), *prog_at(p, q.c[2]), *prog_at(p, q.c[3])};
    if (cls == PC_ROW && !whole) {
        p += r0;
        return vf4{*prog_at(p, q.r[0]), *prog_at(p, q.r[1]), *prog_at(p, q.r[2]), *prog_at(p, q.r[3])};
    }
    const float v = cls == PC_ROW ? *prog_at(p + r0, q.r[0]) : p[0];
    return vf4{v, v, v, v};
}

// ---------------------------------------------------------------------------------------
// elementwise instructions: out = F(a, b, c), or out += F(a, b, c)
// ---------------------------------------------------------------------------------------
template <class F, int NIN, bool ACCUM>
__device__ __forceinline__ void prog_ew_quad(const ProgInstr& in, int64_t e0, int64_t r0, const Pos& q, bool whole,
                                             const float* const (&p)[3], const int (&cls)[3], const F& f) {
    float* out = const_cast<float*>(prog_at(in.out + e0, q.le));
    if (q.n == 4) {
        vf4 v[NIN];
#pragma unroll
        for (int k = 0; k < NIN; ++k) v[k] = prog_quad(p[k], cls[k], e0, r0, q, whole);
        vf4 o = vf4{0.f, 0.f, 0.f, 0.f}, r;
        if (ACCUM) o = ld_c4(out);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float x[3] = {0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < NIN; ++k) x[k] = v[k][j];
            const float fv = f(x);
            r[j] = ACCUM ? o[j] + fv : fv;
        }
        st_c4(out, r);
    } else if (q.n > 0) {
        for (int j = 0; j < q.n; ++j) {
            float x[3] = {0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < NIN; ++k)
                x[k] = prog_val(p[k], cls[k], e0 + q.le + j, r0 + (j == 0 ? q.r[0] : j == 1 ? q.r[1] : q.r[2]),
                                (int32_t)(j == 0 ? q.c[0] : j == 1 ? q.c[1] : q.c[2]));
            const float fv = f(x);
            st_c(out + j, ACCUM ? ld_c(out + j) + fv : fv);
        }
    }
}

template <class F, int NIN, bool ACCUM, int NT>
__device__ __forceinline__ void prog_ew(const ProgInstr& in, const Slab& s, const Pos& first, F f) {
    const float* const p[3] = {in.a, in.b, in.c};
    int cls[3] = {in.cls & 3, (in.cls >> 2) & 3, (in.cls >> 4) & 3};
    if (!(in.flags & PF_ROWDOM)) {
        const bool whole = (s.W & 3) == 0;
        prog_ew_quad<F, NIN, ACCUM>(in, s.e0, s.r0, first, whole, p, cls, f);
        const int32_t cnt = s.rows * s.W;
        for (int32_t le = 4 * (int32_t)threadIdx.x + 4 * NT; le < cnt; le += 4 * NT)
            prog_ew_quad<F, NIN, ACCUM>(in, s.e0, s.r0, prog_pos(s, le), whole, p, cls, f);
    } else {  // over the slab's [rows, 1]: row operands are its elements
#pragma unroll
        for (int k = 0; k < 3; ++k) cls[k] = cls[k] == PC_ROW ? PC_FULL : cls[k];
        for (int32_t le = 4 * (int32_t)threadIdx.x; le < s.rows; le += 4 * NT) {
            Pos q{};
            q.le = (uint32_t)le;
            q.n = s.rows - le < 4 ? s.rows - le : 4;
            prog_ew_quad<F, NIN, ACCUM>(in, s.r0, s.r0, q, true, p, cls, f);
        }
    }
}

// ---------------------------------------------------------------------------------------
// the terms of a gradient that sums over broadcast axes
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ float prog_term(int kind, float u, float v, float d) {
    switch (kind) {  // FBinRg's expressions
        case PT_UG: return u;
        case PT_NEG: return -u;
        case PT_MUL: return u * v;
        case PT_DIV0: return u / v;
        default: return ((-v) / (d * d)) * u;
    }
}
__device__ __forceinline__ int prog_term_operands(int kind) { return kind <= PT_NEG ? 1 : kind <= PT_DIV0 ? 2 : 3; }

// ---------------------------------------------------------------------------------------
// row instructions
// ---------------------------------------------------------------------------------------
// acc = comb(acc, val(c)) over the row's columns in element order, eight loads in flight.
template <class V, class C>
__device__ __forceinline__ float prog_row_serial(int32_t W, float acc, V val, C comb) {
    for (int32_t c = 0; c < W; c += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (c + u < W) v[u] = val(c + u);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (c + u < W) acc = comb(acc, v[u]);
    }
    return acc;
}

// The same across a wavefront, in k_rows_wave's order: lane quads in groups of four, the last W % 4
// elements on the lane after the last quad, then the groups in order and a butterfly.
template <class V, class C>
__device__ __forceinline__ float prog_row_wave(int32_t W, int lane, float init, V val, C comb) {
    const int32_t nq = W >> 2;
    float a4[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) a4[u][j] = init;
    int32_t q = lane;
    for (; q + 192 < nq; q += 256)
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) a4[u][j] = comb(a4[u][j], val(4 * (q + 64 * u) + j));
    for (; q < nq; q += 64)
#pragma unroll
        for (int j = 0; j < 4; ++j) a4[0][j] = comb(a4[0][j], val(4 * q + j));
    if (q == nq)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (4 * q + j < W) a4[0][j] = comb(a4[0][j], val(4 * q + j));
    float acc = init;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = comb(acc, a4[u][j]);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) acc = comb(acc, __shfl_xor(acc, m));
    return acc;
}

struct PAdd {
    __device__ float operator()(float a, float b) const { return a + b; }
};
struct PMax {  // max_simd
    __device__ float operator()(float a, float b) const { return a > b ? a : b; }
};

// MAX / SUM / MEAN over each row, and the un-broadcast of a per-row operand's gradient.
template <int NT>
__device__ __forceinline__ void prog_rows(const ProgInstr& in, const Slab& s) {
    const int op = in.op;
    const int cb = (in.cls >> 2) & 3, cc = (in.cls >> 4) & 3, ca = in.cls & 3;
    const int kind = in.slot, nop = prog_term_operands(kind);
    auto row = [&](int64_t r, int64_t e, bool serial, int lane) {
        if (op == PO_RMAX) {
            auto v = [&](int32_t c) { return ld_c(in.a + e + c); };
            const float m = serial ? prog_row_serial(s.W, -FLT_MAX, v, PMax{}) : prog_row_wave(s.W, lane, -FLT_MAX, v, PMax{});
            if (lane == 0) in.out[r] = m;
        } else if (op == PO_RSUM) {
            auto v = [&](int32_t c) { return ld_c(in.a + e + c); };
            const float m = serial ? prog_row_serial(s.W, 0.0f, v, PAdd{}) : prog_row_wave(s.W, lane, 0.0f, v, PAdd{});
            if (lane == 0) in.out[r] = in.f0 != 0.0f ? m / in.f0 : m;  // MEAN: / f32(W)
        } else {  // PO_RUNB
            auto v = [&](int32_t c) {
                const float u = prog_val(in.a, ca, e + c, r, c);
                const float b = nop > 1 ? prog_val(in.b, cb, e + c, r, c) : 0.0f;
                const float d = nop > 2 ? prog_val(in.c, cc, e + c, r, c) : 0.0f;
                return prog_term(kind, u, b, d);
            };
            if (serial) {
                in.out[r] = prog_row_serial(s.W, in.out[r], v, PAdd{});  // added one at a time, as the serial walk does
            } else {
                const float m = prog_row_wave(s.W, lane, 0.0f, v, PAdd{});
                if (lane == 0) in.out[r] = in.out[r] + m;
            }
        }
    };
    if (s.W <= 64) {
        for (int32_t i = threadIdx.x; i < s.rows; i += NT) row(s.r0 + i, s.e0 + (int64_t)i * s.W, true, 0);
    } else {
        const int lane = threadIdx.x & 63;
        for (int32_t i = threadIdx.x >> 6; i < s.rows; i += NT / 64) row(s.r0 + i, s.e0 + (int64_t)i * s.W, false, lane);
    }
}

// MAX backward over rows of up to 64 (more: the node's own kernel): the row's maximum and its count,
// then out += x == max ? fl(1 / count) * ug : 0. A NaN element is neither the maximum nor counted.
template <int NT>
__device__ __forceinline__ void prog_max_bwd(const ProgInstr& in, const Slab& s, float* sm, float* sg) {
    auto add = [](float& m, uint32_t& c, float v) {
        const bool gt = v > m, eq = v == m;
        c = gt ? 1u : (eq ? c + 1u : c);
        m = gt ? v : m;
    };
    // a row per thread finds (max, factor), then the slab's quads go in flat order
    const int32_t cnt = s.rows * s.W;
    const float* x = in.a + s.e0;
    float* out = in.out + s.e0;
    __syncthreads();  // sm and sg: an instruction of this kind just before may still be read
    for (int32_t i = threadIdx.x; i < s.rows; i += NT) {
        const float* xr = x + (int64_t)i * s.W;
        float m = -FLT_MAX;
        uint32_t n = 0;
        for (int32_t c = 0; c < s.W; c += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (c + u < s.W) v[u] = ld_c(xr + c + u);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (c + u < s.W) add(m, n, v[u]);
        }
        sm[i] = m;
        sg[i] = (1.0f / (float)n) * in.b[s.r0 + i];
    }
    __syncthreads();
    for (int32_t le = 4 * (int32_t)threadIdx.x; le < cnt; le += 4 * NT) {
        if (le + 4 <= cnt) {
            const vf4 xv = ld_c4(x + le), g = ld_c4(out + le);
            int32_t lr = (int32_t)fdiv((uint32_t)le, s.fw), c = le - lr * s.W;
            vf4 r;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                r[j] = g[j] + (xv[j] == sm[lr] ? sg[lr] : 0.0f);
                if (++c == s.W) {
                    c = 0;
                    lr = lr + 1 < s.rows ? lr + 1 : lr;
                }
            }
            st_c4(out + le, r);
        } else {
            for (int32_t i = le; i < cnt; ++i) {
                const int32_t lr = (int32_t)fdiv((uint32_t)i, s.fw);
                st_c(out + i, ld_c(out + i) + (ld_c(x + i) == sm[lr] ? sg[lr] : 0.0f));
            }
        }
    }
}

// SUM / MEAN / MAX over every element, in the one slab that holds them all (up to kProgSingle), in
// the orders of the single kernels: element order up to 64 elements, k_rows_wave's below 2048, else
// chunks of 2048 (k_rows_block's order, 256 threads each) added in chunk order.
__device__ __forceinline__ void prog_all(const ProgInstr& in, const Slab& s, float* ws) {
    const bool rowdom = (in.flags & PF_ROWDOM) != 0;
    const int32_t cnt = rowdom ? s.rows : s.rows * s.W;
    const float* x = in.a + (rowdom ? s.r0 : s.e0);
    const bool mx = in.op == PO_AMAX;
    const float init = mx ? -FLT_MAX : 0.0f;
    auto comb = [mx](float a, float b) { return mx ? (a > b ? a : b) : a + b; };
    auto val = [x](int32_t c) { return ld_c(x + c); };
    const int t = threadIdx.x;
    float acc = init;
    if (cnt <= 64) {
        if (t == 0) acc = prog_row_serial(cnt, init, val, comb);
    } else if (cnt < 2048) {
        if (t < 64) acc = prog_row_wave(cnt, t, init, val, comb);
    } else {
        constexpr int32_t kChunk = 2048, kT = 256;
        static_assert(kProgSingle <= 4 * kChunk, "a chunk for each quarter of the workgroup");
        const int32_t s0 = (t / kT) * kChunk, tt = t % kT;
        if (s0 < cnt) {
            const int32_t len = cnt - s0 < kChunk ? cnt - s0 : kChunk, nq = len >> 2;
            float a2[2][4];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    a2[u][j] = init;
                    if (tt + u * kT < nq) a2[u][j] = comb(init, val(s0 + 4 * (tt + u * kT) + j));
                }
            if (tt < (len & 3)) a2[1][3] = comb(a2[1][3], val(s0 + 4 * nq + tt));
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc = comb(acc, a2[u][j]);
#pragma unroll
            for (int m = 32; m >= 1; m >>= 1) acc = comb(acc, __shfl_xor(acc, m));
        }
        if ((t & 63) == 0) ws[t >> 6] = acc;
        __syncthreads();
        if (t == 0) {
            acc = init;
            for (int c = 0; c * kChunk < cnt; ++c)
                acc = comb(acc, comb(comb(comb(ws[4 * c], ws[4 * c + 1]), ws[4 * c + 2]), ws[4 * c + 3]));
        }
        __syncthreads();  // ws is used again by the next instruction of this kind
    }
    if (t == 0) in.out[0] = in.f0 != 0.0f ? acc / in.f0 : acc;
}

// The un-broadcast of a per-column operand's gradient over the slab's rows, one wavefront per 64
// columns: a lane per column (W >= 64), or 64 / P lanes per column taking rows in turn (P the power
// of two that holds W), whose sums a butterfly adds. One slab of up to 64 rows: a lane walks its
// column's rows in order, adding into the gradient one at a time (the single kernels' order).
__device__ __forceinline__ void prog_cols(const ProgInstr& in, const Slab& s, float* part, bool single, int32_t chunk,
                                          int lane) {
    const int kind = in.slot, nop = prog_term_operands(kind);
    const int ca = in.cls & 3, cb = (in.cls >> 2) & 3, cc = (in.cls >> 4) & 3;
    const bool serial = single && s.rows <= 64;
    int P = 64;
    if (!serial && s.W < 64)
        while (P / 2 >= s.W) P /= 2;
    const int G = 64 / P;
    const int32_t c = chunk * 64 + (lane & (P - 1));
    const bool live = c < s.W;
    // an operand's element at row rr: base[rr * stride]
    auto base = [&](const float* p, int cls) {
        return p + (cls == PC_FULL ? s.e0 + c : cls == PC_ROW ? s.r0 : cls == PC_COL ? (int64_t)c : 0);
    };
    auto stride = [&](int cls) { return cls == PC_FULL ? s.W : cls == PC_ROW ? 1 : 0; };
    float acc = serial && live ? in.out[c] : 0.0f;
    if (live) {
        const float *pa = base(in.a, ca), *pb = nop > 1 ? base(in.b, cb) : pa, *pd = nop > 2 ? base(in.c, cc) : pa;
        const int32_t sa = stride(ca), sb = nop > 1 ? stride(cb) : sa, sd = nop > 2 ? stride(cc) : sa;
        constexpr int U = 16;
        for (int32_t r = lane / P; r < s.rows; r += U * G) {
            float u[U], v[U], d[U];
#pragma unroll
            for (int k = 0; k < U; ++k) {  // a row past the slab reads its last one, unused
                const int32_t rr = r + k * G < s.rows ? r + k * G : s.rows - 1;
                u[k] = pa[(int64_t)rr * sa];
            }
            if (nop > 1)
#pragma unroll
                for (int k = 0; k < U; ++k) v[k] = pb[(int64_t)(r + k * G < s.rows ? r + k * G : s.rows - 1) * sb];
            if (nop > 2)
#pragma unroll
                for (int k = 0; k < U; ++k) d[k] = pd[(int64_t)(r + k * G < s.rows ? r + k * G : s.rows - 1) * sd];
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const float t = acc + prog_term(kind, u[k], v[k], d[k]);
                acc = r + k * G < s.rows ? t : acc;
            }
        }
    }
    for (int m = 32; m >= P; m >>= 1) acc = acc + __shfl_xor(acc, m);
    if (live && lane < P) {
        if (!single) part[(int64_t)blockIdx.x * s.W + c] = acc;
        else in.out[c] = serial ? acc : in.out[c] + acc;
    }
}

// ---------------------------------------------------------------------------------------
// the program
// ---------------------------------------------------------------------------------------
template <int NT>
__global__ void __launch_bounds__(NT)
    k_prog(const ProgInstr* __restrict__ prog, int na, int nb, int64_t R, int32_t W, FastDiv fw, int32_t rpw, float* part) {
    __shared__ float sm[kProgRows], sg[kProgRows], ws[NT / 64];
    const bool single = gridDim.x == 1;
    Slab s;
    s.r0 = (int64_t)blockIdx.x * rpw;
    s.rows = (int32_t)(R - s.r0 < rpw ? R - s.r0 : rpw);
    s.e0 = s.r0 * W;
    s.W = W;
    s.fw = fw;
    const Pos first = prog_pos(s, 4 * (int32_t)threadIdx.x);
    const Slab whole_slab = s;
    ProgInstr nxt = prog[0];
    for (int i = 0; i < na; ++i) {
        const ProgInstr in = nxt;
        if (i + 1 < na + nb) nxt = prog[i + 1];
        if (in.flags & PF_BARRIER) __syncthreads();
        // opaque per instruction: hoisted out of the loop, what each kind derives from the slab's
        // shape filled the scalar registers and was spilled and read back by every instruction
        s = whole_slab;
        asm volatile("" : "+s"(s.rows), "+s"(s.W));
#define MH_EW(OPC, F, NIN, ACC, ...) \
    case OPC: prog_ew<F, NIN, ACC, NT>(in, s, first, F __VA_ARGS__); break
        switch (in.op) {
            MH_EW(PO_ADD, FBin<MH_ADD>, 2, false, {});
            MH_EW(PO_SUB, FBin<MH_SUB>, 2, false, {});
            MH_EW(PO_MUL, FBin<MH_MUL>, 2, false, {});
            MH_EW(PO_DIV, FBin<MH_DIV>, 2, false, {});
            MH_EW(PO_EXP, FUn<MH_EXP>, 1, false, {});
            MH_EW(PO_LOG, FUn<MH_LOG>, 1, false, {});
            MH_EW(PO_SIGMOID, FUn<MH_SIGMOID>, 1, false, {});
            MH_EW(PO_RELU, FUn<MH_RELU>, 1, false, {});
            MH_EW(PO_TANH, FUn<MH_TANH>, 1, false, {});
            MH_EW(PO_LEAKY, FLeaky, 1, false, {in.f0});
            MH_EW(PO_CLIP, FClip, 1, false, {in.f0, in.f1});
            MH_EW(PO_G_UG, FProgUg, 1, true, {});
            MH_EW(PO_G_NEG, FProgNeg, 1, true, {});
            MH_EW(PO_G_MUL, FProgMul, 2, true, {});
            MH_EW(PO_G_DIV0, FProgDiv0, 2, true, {});
            MH_EW(PO_G_DIV1, FProgDiv1, 3, true, {});
            MH_EW(PO_G_EXP, FUnBwd<MH_EXP>, 2, true, {});
            MH_EW(PO_G_LOG, FUnBwd<MH_LOG>, 2, true, {});
            MH_EW(PO_G_SIGMOID, FUnBwd<MH_SIGMOID>, 2, true, {});
            MH_EW(PO_G_RELU, FUnBwd<MH_RELU>, 2, true, {});
            MH_EW(PO_G_TANH, FUnBwd<MH_TANH>, 2, true, {});
            MH_EW(PO_G_LEAKY, FLeakyBwd, 2, true, {in.f0});
            MH_EW(PO_G_CLIP, FClipBwd, 2, true, {in.f0, in.f1});
            MH_EW(PO_G_SCALE, FScaleBcast<false>, 1, true, {in.f0});
            case PO_RMAXB: prog_max_bwd<NT>(in, s, sm, sg); break;
            case PO_ASUM:
            case PO_AMAX:
                if constexpr (NT == 1024) prog_all(in, s, ws);  // one slab only
                break;
            default: prog_rows<NT>(in, s); break;
        }
#undef MH_EW
    }
    if (nb > 0) {
        __syncthreads();
        const int32_t chunks = (W + 63) / 64;
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        for (int u = wave; u < nb * chunks; u += NT / 64) {
            const int k = u / chunks;
            const ProgInstr in = prog[na + k];
            prog_cols(in, s, part + in.part, single, u - k * chunks, (int)(threadIdx.x & 63));
        }
    }
}

// The slabs' partials of each sum (grid y), added in slab order over 32 groups, folded as a tree:
// out += sum.
__global__ void __launch_bounds__(256)
    k_prog_final(const ProgSum* __restrict__ sums, const float* __restrict__ part, int32_t nwg) {
    constexpr int G = 32, Q = 256 / G;
    __shared__ float lds[G][Q];
    const ProgSum t = sums[blockIdx.y];
    const int q = threadIdx.x % Q, g = threadIdx.x / Q;
    const int32_t c = blockIdx.x * Q + q;
    if ((int32_t)(blockIdx.x * Q) >= t.ncol) return;  // uniform over the block
    float acc = 0.0f;
    if (c < t.ncol) {
        const int32_t per = (nwg + G - 1) / G, w0 = g * per, w1 = w0 + per < nwg ? w0 + per : nwg;
        const float* p = part + t.part;
        for (int32_t w = w0; w < w1; w += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = w + u < w1 ? p[(int64_t)(w + u) * t.ncol + c] : 0.0f;
#pragma unroll
            for (int u = 0; u < 8; ++u) acc = acc + v[u];
        }
    }
    lds[g][q] = acc;
    __syncthreads();
#pragma unroll
    for (int h = G / 2; h >= 1; h >>= 1) {
        if (g < h) lds[g][q] = lds[g][q] + lds[g + h][q];
        __syncthreads();
    }
    if (g == 0 && c < t.ncol) t.out[c] = t.out[c] + lds[0][q];
}

int prog_launch(const ProgRun& p) {
    MH_TRACE("mh_model_program");  // stands for its nodes' own ranges
    hipStream_t st = ctx().stream;
    const FastDiv fw = make_fastdiv((uint32_t)p.W);
    if (p.nwg == 1)
        hipLaunchKernelGGL(k_prog<1024>, dim3(1), dim3(1024), 0, st, p.prog, p.na, p.nb, p.R, p.W, fw, p.rpw, p.part);
    else
        hipLaunchKernelGGL(k_prog<256>, dim3((unsigned)p.nwg), dim3(256), 0, st, p.prog, p.na, p.nb, p.R, p.W, fw, p.rpw,
                           p.part);
    if (p.nwg > 1 && p.nsums > 0)
        hipLaunchKernelGGL(k_prog_final, dim3((unsigned)((p.maxcol + 7) / 8), (unsigned)p.nsums), dim3(256), 0, st, p.sums,
                           p.part, p.nwg);
    return MH_OK;
}

}  // namespace mh
