// Fully connected GEMMs on the bf16 matrix cores with every fp32 operand split
// exactly into three bf16 pieces (fc_split.hip).
#pragma once

#include "conv_common.hpp"

namespace ach {

// out[r][c] = sum over k of A(r, k) * B(c, k), r < R (the batch, or filters),
// c < N.  An operand is row-major P[r][k] or k-major P[k][r].
struct FcOperand {
    const float *p;
    int rows;
    bool kmajor;
};

// whether the forward or input-gradient form takes this path, and the K
// slices it splits into (at most room)
int fc_split_slices(int batch, int features, int K, int room);
// y[r][c] or, with slices > 1, part[z][r][c]; the epilogue e (of feature c)
// applies when slices == 1
int fc_split_launch(const FcOperand &a, const FcOperand &b, int K, int slices, float *y,
                    float *part, const Epi &e, hipStream_t st);

bool fc_split_wgrad(int F, int C, int batch);
// dw[f][c] += sum over b of dy[b][f] * x[b][c], then the SGD step when sg.w
int fc_split_wgrad_launch(int F, int C, int batch, const float *dy, const float *x, float *dw,
                          const Sgd &sg, hipStream_t st);

}  // namespace ach
