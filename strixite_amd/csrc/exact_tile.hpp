// Exact-weight projections on 16-row tiles (exact_tile.hip): dense Q4 / Q8 at small batches, and every expert and dense
// projection with FP32 activations or Q5 weights. Internal entries of the launchers in experts.hip.
#pragma once

#include "strixite_moe.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>

namespace strix::kernels::xt {

enum Mode { DENSE = 0, GROUPED = 1, PERSLOT = 2 };

struct Args {
    const void *x;                        // activation rows [*, K] (FP32 or BF16)
    const uint8_t *q;
    const uint16_t *scale, *minv;
    int64_t N, K, G;                      // N: weight rows an expert (DENSE: all)
    int64_t E, A, S;                      // S: output rows (DENSE: M tokens; slots otherwise); x row of a slot: slot / A
    const int32_t *ws, *ids;              // GROUPED: the grouping workspace; PERSLOT: ids [S]
    uint32_t *err;                        // PERSLOT: the expert error word
    void *y;                              // output [S, ldy] in the output dtype
    int64_t ldy;
    int64_t ncol;                         // output columns (SwiGLU: I = N / 2)
};

// y = x W^T (swiglu: silu(gate) * up of the expert's rows j and ncol + j). fmt: 4, 5 or 8 (the code bits)
void project(int fmt, Mode mode, bool swiglu, Act x_act, Act y_act, const Args &a, hipStream_t stream);

// y [M, ncol] = sum over the token's A slots, in order with fmaf, of coef[slot] (x[slot] . W[ids[slot]]); an invalid id:
// NaN row and the error word. x rows are slots; a.S = M; x and y share a dtype.
void perslot_combine(int fmt, Act act, const Args &a, const float *coef, hipStream_t stream);

// One token's down, combine and residual in one launch (Q4 or Q8 experts, BF16, at most kOneTokenSlots slots): y [ncol] =
// sum over the slots, in order with fmaf, of coef[slot] (x[slot] . W[ids[slot]]), rounded to BF16 once; out (optional) =
// resid + y. An invalid id: NaN. a.x: h [A, K], a.ids [A], a.y: y.
constexpr int64_t kOneTokenSlots = 16;
void one_token_down(int fmt, const Args &a, const float *coef, const uint16_t *resid, uint16_t *out, hipStream_t stream);

}  // namespace strix::kernels::xt
