// The sublayer tail with its folded projection for few rows (ffn_small.hip), launched by the entry points of ffn_fused.hip.
#pragma once

#include "common.h"

namespace bnb {

struct FfnSmallArgs {
    const float *x;
    int64_t x_stride;
    const uint16_t *rows_a;
    int64_t rows_a_stride;
    const uint16_t *rows_b;  // NULL: rows_a is projected as it is
    int64_t rows_b_stride;
    const uint16_t *wproj;
    const float *norm_w;
    float eps;
    const uint16_t *wpack;
    float *out;
    int64_t R;
    const float *next_norm_w;
    float next_eps;
    const uint16_t *next_wpack;
    uint16_t *next_out;  // NULL: no head
    int next_features;
    float *s_out;  // the update's form (rows_b and next_out NULL): the residual sum and the normalised rows leave as well
    uint16_t *n_out;
};

// Rows up to which the split form is the faster one.
int64_t ffn_small_rows_limit();

int launch_ffn_small(const FfnSmallArgs &a, hipStream_t s);

}  // namespace bnb
