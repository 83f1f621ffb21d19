// mh_functors.h -- the per-element functions of Mantle's ops, forward and backward, in the
// reference's expression order: shared by the elementwise engines and the executor's program
// kernel, so that a value has the same bits in both.
#pragma once

#include "mh_internal.h"
#include "mh_math.h"

namespace mh {

struct DevScal {
    const float* p[4];
};

template <int N>
struct InPtrs {
    const float* p[N > 0 ? N : 1];
};

// ---------------------------------------------------------------------------------------
// functors: operator()(v) with v[k] the k-th input value; setup() reads device scalars.
// ---------------------------------------------------------------------------------------
template <int OP>
struct FBin {  // add/sub/mul/div, math_util.mojo:37-126
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const {
        if constexpr (OP == MH_ADD) return v[0] + v[1];
        else if constexpr (OP == MH_SUB) return v[0] - v[1];
        else if constexpr (OP == MH_MUL) return v[0] * v[1];
        else return v[0] / v[1];
    }
};

template <int OP>
struct FUn {  // elwise_transform bodies
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const {
        if constexpr (OP == MH_EXP) return mexp(v[0]);
        else if constexpr (OP == MH_LOG) return mlog(v[0]);
        else if constexpr (OP == MH_SIGMOID) return msigmoid(v[0]);
        else if constexpr (OP == MH_RELU) return mrelu(v[0]);
        else return mtanh(v[0]);
    }
};

struct FPowi {  // POW.forward: powi(x, Int(t2[0])), basics.mojo:320-327
    int64_t n;
    __device__ void setup(const DevScal& s) {
        float e = s.p[0][0];
        n = (e != e) ? 0 : (int64_t)__builtin_truncf(e);
    }
    __device__ float operator()(const float* v) const { return mpowi(v[0], n); }
};

struct FPowiN {  // elwise_pow with its integer exponent given, tensorutils.mojo:226-239
    int64_t n;
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const { return mpowi(v[0], n); }
};

template <int OP>
struct FUnBwd {  // v[0] = x, v[1] = ug: the rg of each unary struct backward
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const {
        const float x = v[0], ug = v[1];
        if constexpr (OP == MH_EXP) return mexp(x) * ug;  // basics.mojo:281-284
        else if constexpr (OP == MH_LOG) return ug / x;   // basics.mojo:305-309
        else if constexpr (OP == MH_SIGMOID) {            // mlops.mojo:50-76
            float s = msigmoid(x);
            return (s * (1.0f - s)) * ug;
        } else if constexpr (OP == MH_RELU) {             // mlops.mojo:99-125
            return (x > 0.0f ? 1.0f : 0.0f) * ug;
        } else {                                          // mlops.mojo:209-235
            float t = mtanh(x);
            return (1.0f - t * t) * ug;
        }
    }
};

struct FPowBwdX {  // basics.mojo:345-357: (a * (x + 1e-12) ** (a - 1)) * ug
    float a, am1;
    __device__ void setup(const DevScal& s) {
        a = s.p[0][0];
        am1 = a - 1.0f;
    }
    __device__ float operator()(const float* v) const { return (a * mpowf(v[0] + 1e-12f, am1)) * v[1]; }
};

// Binary struct backward of one operand (basics.mojo:28-219). Inputs: v[0] = ug, then
//   ADD, SUB id0: -            -> ug
//   SUB id1:      -            -> ug * -1
//   MUL id0:      v[1] = t2    -> ug * t2        MUL id1: v[1] = t1 -> ug * t1
//   DIV id0:      v[1] = t2    -> ug / t2
//   DIV id1:      v[1] = t1, v[2] = t2 -> ((-t1) / (t2 * t2)) * ug
//   DIV id1 with t2 of shape (1) (DIVS): v[1] = t1, f = -1 / (s * s) -> (f * t1) * ug
template <int OP, int ID, bool DIVS>
struct FBinRg {
    float f;
    __device__ void setup(const DevScal& s) {
        if constexpr (DIVS) {
            const float t = s.p[0][0];
            f = -1.0f / (t * t);
        }
    }
    __device__ float operator()(const float* v) const {
        const float ug = v[0];
        if constexpr (OP == MH_ADD) return ug;
        else if constexpr (OP == MH_SUB) return ID == 0 ? ug : ug * -1.0f;
        else if constexpr (OP == MH_MUL) return ug * v[1];
        else if constexpr (ID == 0) return ug / v[1];
        else if constexpr (DIVS) return (f * v[1]) * ug;
        else return ((-v[1]) / (v[2] * v[2])) * ug;
    }
};

// FBinRg's expressions over the operands they read: v[0] = ug, v[1], v[2].
struct FProgUg {
    __device__ float operator()(const float* v) const { return v[0]; }
};
struct FProgNeg {
    __device__ float operator()(const float* v) const { return v[0] * -1.0f; }
};
struct FProgMul {
    __device__ float operator()(const float* v) const { return v[0] * v[1]; }
};
struct FProgDiv0 {
    __device__ float operator()(const float* v) const { return v[0] / v[1]; }
};
struct FProgDiv1 {
    __device__ float operator()(const float* v) const { return ((-v[1]) / (v[2] * v[2])) * v[0]; }
};

// SUM/MEAN axis backward (basics.mojo:416-425, 489-506): fill(c) then accumulate_op[mul]
// with the broadcast ug: rg = c * ug; TWICE (rg = (c * ug) * ug) when the reduced shape
// equals the input shape (accumulate_op applies func twice then, tensorutils.mojo:380-393).
template <bool TWICE>
struct FScaleBcast {
    float c;
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const {
        if constexpr (TWICE) return (c * v[0]) * v[0];
        else return c * v[0];
    }
};

// MEAN all-element backward (basics.mojo:470-487): g = f32(1/N) * ug[0], filled.
struct FMeanAll {
    float c, g;
    __device__ void setup(const DevScal& s) { g = c * s.p[0][0]; }
    __device__ float operator()(const float*) const { return g; }
};

// MAX backward routing (basics.mojo:567-577, 597-613): v[0] = x, v[1] = line max,
// v[2] = fl(1/count) of the line, v[3] = ug of the line.
struct FMaxRoute {
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const { return v[0] == v[1] ? v[2] * v[3] : 0.0f; }
};

// Accumulating functors whose contribution is +0 almost everywhere: the engines store a quad
// only when its bits change (bits_differ4), which leaves memory exactly as storing every quad
// would, without writing back the untouched ones.
template <class F>
inline constexpr bool kSparseAccum = false;
template <>
inline constexpr bool kSparseAccum<FMaxRoute> = true;

struct FFma {  // FMA.forward, basics.mojo:782-786: t1.fma(t2, t3), a single rounding
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const { return __builtin_fmaf(v[0], v[1], v[2]); }
};

struct FLeaky {  // LEAKYRELU.forward, mlops.mojo:141-154
    float slope;
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const { return v[0] > 0.0f ? v[0] : v[0] * slope; }
};

struct FLeakyBwd {  // v[0] = x, v[1] = ug: LEAKYRELU.backward, mlops.mojo:164-184
    float slope;
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const { return (v[0] > 0.0f ? 1.0f : slope) * v[1]; }
};

// min / max as LLVM minnum / maxnum: a NaN operand yields the other one, equal operands the
// first, so a NaN input clips to hi.
__device__ __forceinline__ float minnum_f(float a, float b) { return (b < a || a != a) ? b : a; }
__device__ __forceinline__ float maxnum_f(float a, float b) { return (b > a || a != a) ? b : a; }

struct FClip {  // CLIP.forward, mlops.mojo:243-266: max(min(x, hi), lo)
    float lo, hi;
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const { return maxnum_f(minnum_f(v[0], hi), lo); }
};

struct FClipBwd {  // v[0] = x, v[1] = ug: CLIP.backward, mlops.mojo:281-297
    float lo, hi;
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const { return (v[0] >= lo && v[0] <= hi) ? v[1] : 0.0f; }
};

template <int ID>
struct FFmaRg {  // FMA.backward, basics.mojo:804-817: id 0 ug * t2, id 1 ug * t1, id 2 ug
    __device__ void setup(const DevScal&) {}
    __device__ float operator()(const float* v) const {
        if constexpr (ID == 2) return v[0];
        else return v[0] * v[1];
    }
};

}  // namespace mh
