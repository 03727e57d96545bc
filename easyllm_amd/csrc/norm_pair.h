// RMSNorm for the whole-layer calls (layer.cpp; defined in norm.hip): the forward that writes its sum twice, the backward in two parts.
#pragma once
#include "common.h"

// Per-block partial sums of one norm weight's gradient, `blocks` rows of h floats, and where their sum goes (one of f32 / bf16).
struct NormWeightGrad {
    const float* partials;
    void *bf16, *f32;
    int accumulate, blocks;
};

// ezl_rmsnorm_fwd with a residual, the sum also to sum_copy (null, or 16-byte aligned and none of the other tensors)
__attribute__((visibility("hidden"))) int rmsnorm_fwd_keep_sum(const void* x, const void* residual, const void* weight, void* y, void* sum_out,
                                                               void* sum_copy, void* rstd, int64_t rows, int64_t h, float eps, void* stream);

// ezl_rmsnorm_bwd up to the partial sums, which it leaves in `workspace` (as large as there)
__attribute__((visibility("hidden"))) int rmsnorm_bwd_rows(const void* dy, const void* x, const void* weight, const void* rstd, const void* dresidual,
                                                           void* dx, void* dw_bf16, void* dw_f32, int accumulate, void* workspace, int64_t rows,
                                                           int64_t h, NormWeightGrad& grad, void* stream);
// the sums of two norms of one width, in one launch
__attribute__((visibility("hidden"))) int norm_weight_grads(const NormWeightGrad& a, const NormWeightGrad& b, int64_t h, void* stream);
