// Products over one reduction length in one launch, for the whole-layer calls (layer.cpp; defined in gemm.hip).
#pragma once
#include "common.h"

constexpr int kGemmListMax = 7;  // the weight gradients of a decoder layer: q, k, v, o, gate, up, down

// Workspace of C[i] (=|+=) A[i] * B[i], i < sum of counts, as one launch; -1 where the products are estimated to be faster in
// `pieces` pieces of counts[p] consecutive ones, each in one launch or one by one.  beyond_cache: only as 256 x 256 tiles.
__attribute__((visibility("hidden"))) int64_t gemm_list_workspace_bytes(int pieces, const int* counts, const int64_t* M, const int64_t* N,
                                                                        int64_t K, bool beyond_cache);
// as ezl_gemm_bf16_group, for up to kGemmListMax products
__attribute__((visibility("hidden"))) int gemm_list(int count, const void* const* A, const void* const* B, void* const* C, const int64_t* M,
                                                    const int64_t* N, int64_t K, const int64_t* lda, const int64_t* ldb, const int64_t* ldc,
                                                    int a_kc, int b_kc, int out_dtype, const int* accumulate, void* workspace,
                                                    int64_t workspace_bytes, void* stream);

// C[M, N] += A[M, K] * B[N, K]^T, all contiguous bf16, the product rounded to bf16 before it is added: the bits of a product and an addition
__attribute__((visibility("hidden"))) int gemm_forward_add(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, void* workspace,
                                                           int64_t workspace_bytes, void* stream);
