// mh_program.h -- the executor's programs: instructions, and a run of them (mh_program.hip).
#pragma once

#include "mh_internal.h"

namespace mh {

// An operand's form in the [R, W] view.
enum ProgCls : int { PC_FULL = 0, PC_ROW = 1, PC_COL = 2, PC_SCAL = 3 };

enum ProgOp : int {
    PO_ADD, PO_SUB, PO_MUL, PO_DIV, PO_EXP, PO_LOG, PO_SIGMOID, PO_RELU, PO_TANH, PO_LEAKY, PO_CLIP,
    // out += the gradient of an operand of the output's own form: a = ug, then its other operands
    PO_G_UG, PO_G_NEG, PO_G_MUL, PO_G_DIV0, PO_G_DIV1,
    // out += a unary op's gradient: a = x, b = ug
    PO_G_EXP, PO_G_LOG, PO_G_SIGMOID, PO_G_RELU, PO_G_TANH, PO_G_LEAKY, PO_G_CLIP,
    PO_G_SCALE,        // out += f0 * a (SUM / MEAN backward)
    PO_RMAX, PO_RSUM,  // over each row (f0: MEAN's divisor, or 0)
    PO_RUNB,           // out (per row) += the row's sum of a gradient's terms (kind in slot)
    PO_RMAXB,          // MAX backward: a = x, b = ug per row
    PO_ASUM, PO_AMAX,  // over every element (f0: MEAN's divisor, or 0)
    PO_CUNB            // out (per column) += the column's sum of a gradient's terms (kind in slot)
};
enum ProgTerm : int { PT_UG = 0, PT_NEG = 1, PT_MUL = 2, PT_DIV0 = 3, PT_DIV1 = 4 };

constexpr int PF_ROWDOM = 1;   // over the slab's [rows, 1] rather than its elements
constexpr int PF_BARRIER = 2;  // a barrier before this instruction

struct ProgInstr {
    int32_t op, cls, flags, slot;
    float f0, f1;
    int64_t part;  // first float of this sum's partials
    float* out;
    const float *a, *b, *c;
};
struct ProgSum {
    float* out;
    int64_t part;
    int32_t ncol, pad;
};

constexpr int kProgRows = 1024;          // rows of a slab at most, where there are several or a MAX gradient
constexpr size_t kProgMaxSums = 4096;    // sums over rows of one program
constexpr int64_t kProgSingle = 8192;   // elements up to which one workgroup runs the whole view

constexpr int64_t kProgMax = (int64_t)1 << 20;

struct ProgRun {
    const ProgInstr* prog = nullptr;  // device: na instructions in order, then nb sums over rows
    const ProgSum* sums = nullptr;    // device
    float* part = nullptr;
    int na = 0, nb = 0, nsums = 0, maxcol = 0;
    int64_t R = 0;
    int32_t W = 0, rpw = 0, nwg = 0;
};
int prog_launch(const ProgRun& p);

}  // namespace mh
