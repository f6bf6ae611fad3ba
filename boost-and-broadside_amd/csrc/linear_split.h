// The float32 Linear on three-piece bf16 operands (linear_split.hip), checked and called from linear_f32.hip.
#pragma once

#include "common.h"

namespace bnb {

struct LinearSplitArgs {
    const float *x;
    int64_t x_stride;
    const float *x2;  // gelu(x) * x2 when given
    int64_t x2_stride;
    const float *norm_w;  // rmsnorm(x) * norm_w when given (K == 128)
    float eps;
    const uint16_t *w;  // [fb][K/128][ks][piece][lane][8], fb < n_blocks
    const float *bias, *resid;
    int64_t resid_stride;
    float *out;
    int64_t out_stride, R;
    int K, n_blocks;
};

int launch_linear_split(const LinearSplitArgs &args, bool gate, hipStream_t stream);

}  // namespace bnb
