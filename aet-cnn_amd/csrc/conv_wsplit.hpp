// Weight gradient of 3x3 stride-1 "same" convolutions on the bf16 matrix cores
// with every fp32 operand split exactly into three bf16 pieces
// (conv_wsplit.hip).
#pragma once

#include "conv_common.hpp"

namespace ach {

struct WsplitPlan {
    bool ok;     // the geometry takes this path
    int splits;  // K slices: partial sums part[z][k*k][F][C]
    int spw;     // K steps per (slice, group)
};

// what the fp32 kernel would do: parts of K, the additions that one of them
// goes through when they are added up (in groups), and its modelled time
struct Fp32Wgrad {
    int parts, adds;
    double us;
};

// room: slices of partial sums that the caller's workspace holds
WsplitPlan wsplit_plan(const ConvGeom &g, const Fp32Wgrad &fp32, int room);

// part[z][ki*k + kj][f][c] = the slice's sums of dy * shifted x
int wsplit_launch(const ConvGeom &g, const WsplitPlan &pl, const float *x, const float *dy,
                  float *part, hipStream_t st);

// dw += the slices' sums in a fixed order, then the SGD step when sg.w
int wsplit_reduce(const ConvGeom &g, const WsplitPlan &pl, const float *part, float *dw,
                  const Sgd &sg, hipStream_t st);

}  // namespace ach
