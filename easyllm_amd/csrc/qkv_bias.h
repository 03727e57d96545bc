// Biases of a layer's q / k / v projections in the whole-layer calls (layer.cpp; kernels in elementwise.hip).
#pragma once
#include "common.h"

struct QkvBiasGrad {  // per projection: fp32 target (accumulate: added to), else bf16 target, else none
    float* f32[3];
    bf16_t* bf16[3];
    int accumulate[3];
};

// out_i = x_i + bias_i (rounded to bf16), then q and k rotated: rows of nq, nk and nk heads of d, contiguous
__attribute__((visibility("hidden"))) int qkv_bias_rope(const void* const* x, const void* const* bias, void* const* out, int64_t nq, int64_t nk,
                                                        int64_t d, const void* cos_table, const void* sin_table, const void* position_ids,
                                                        int64_t s, int64_t b, int64_t npos, hipStream_t stream);
// column sums of dq | dk | dv in rows of qw + 2 kw; workspace: ezl_bias_grad_workspace_bytes(rows, qw + 2 kw)
__attribute__((visibility("hidden"))) int qkv_bias_grad(const void* dqkv, const QkvBiasGrad& g, int64_t rows, int64_t qw, int64_t kw,
                                                        void* workspace, hipStream_t stream);
