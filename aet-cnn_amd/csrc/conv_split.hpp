// Forward / stride-1 input-gradient convolution on the bf16 matrix cores with
// every fp32 operand split exactly into three bf16 pieces (conv_split.hip).
#pragma once

#include "conv_common.hpp"

namespace ach {

struct SplitFwdPlan {
    bool ok;        // the geometry takes this path
    int wm, wn, kg; // waves along M and N of one K group, K groups
    int tpt;        // staging tasks per thread (compile-time cap)
    int nbuf;       // LDS patch buffers
    int npx;        // patch pixels reserved
    int splits;     // grid slices of K (each kg groups wide); partials if > 1
};

// what the fp32 kernel would do: parts of K that it adds up, slices of partial
// sums that it writes, tiles of its grid and k-tiles of a part
struct Fp32Fwd {
    int parts, slices, tiles, ktiles;
};

// kg_ok: the call may run two K groups per workgroup; room: the slices of
// partial sums that the caller's workspace holds
SplitFwdPlan split_fwd_plan(const ConvGeom &g, bool kg_ok, const Fp32Fwd &fp32, int room);

// y (or part[z][m][n] when pl.splits > 1) = conv(x, wt); wt k-major Wt[K][M].
// The epilogue e is applied when K is not split over the grid.
int split_fwd_launch(const ConvGeom &g, const SplitFwdPlan &pl, const float *x, const float *wt,
                     float *y, float *part, const Epi &e, hipStream_t st);

}  // namespace ach
