// Optimizer step for the parameters of the decoder stack on gfx950 (HBM-bound): fp32 master weights, fp32 gradient
// buffers, bf16 model weights.
//
// Restates what the reference's Megatron path runs after backward: apex `FusedAdam` in its default AdamW mode
// (built at llm/utils/model/optimizer_helper.py:93-95 from configs/megatron/llama_7b_sft.yaml:106-112) under
// DeepSpeed's bf16 optimizer with `gradient_clipping: 1.0` (llama_7b_sft.yaml:13): global L2 norm of all gradients,
// clip coefficient max_norm / (norm + 1e-6) applied when below one, then per element
//     m = b1 m + (1 - b1) g;  v = b2 v + (1 - b2) g^2;  p -= lr (m / bc1 / (sqrt(v / bc2) + eps) + wd p)
// with bc = 1 - beta^step, and the bf16 weight refreshed from the fp32 master value.
// The norm is reduced in a fixed order (per-block partials, then one block), so a step is bit-reproducible; the clip
// coefficient stays on the device: nothing here synchronises with the host.
#include "common.h"

namespace {

constexpr int kOptBlock = 256;
constexpr int kSumsqPartials = 256;  // partial sums written per ezl_sumsq_f32 call

// partials[b] = sum of x[i]^2 over block b's share (grid-stride over 4-float vectors, four loads in flight per thread,
// tail by block 0)
constexpr int kSumsqBlock = 1024;
__global__ __launch_bounds__(kSumsqBlock) void sumsq_partial_kernel(const float* __restrict__ x, int64_t n, float* __restrict__ partials) {
    __shared__ float red[kSumsqBlock / 64];
    const int64_t n4 = n >> 2;
    const int64_t stride = (int64_t)gridDim.x * kSumsqBlock;
    float acc = 0.f;
    int64_t i = (int64_t)blockIdx.x * kSumsqBlock + threadIdx.x;
    for (; i + 3 * stride < n4; i += 4 * stride) {
        f32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = reinterpret_cast<const f32x4*>(x)[i + u * stride];
#pragma unroll
        for (int u = 0; u < 4; ++u) acc += v[u][0] * v[u][0] + v[u][1] * v[u][1] + v[u][2] * v[u][2] + v[u][3] * v[u][3];
    }
    for (; i < n4; i += stride) {
        const f32x4 v = reinterpret_cast<const f32x4*>(x)[i];
        acc += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
        const float v = x[(n4 << 2) + threadIdx.x];
        acc += v * v;
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < kSumsqBlock / 64; ++k) t += red[k];
        partials[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(256) void zero_f32_kernel(float* __restrict__ x, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) x[i] = 0.f;
}

// out[0] = sqrt(sum partials), out[1] = clip coefficient: max_norm / (norm + 1e-6) if that is below one, else 1
__global__ __launch_bounds__(1024) void clip_coef_kernel(const float* __restrict__ partials, int64_t count, float max_norm,
                                                         float* __restrict__ out) {
    __shared__ double red[16];
    double acc = 0.0;
    for (int64_t i = threadIdx.x; i < count; i += 1024) acc += (double)partials[i];
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int i = 0; i < 16; ++i) t += red[i];
        const float norm = (float)sqrt(t);
        float coef = 1.0f;
        if (max_norm > 0.f) {
            const float c = max_norm / (norm + 1e-6f);
            if (c < 1.0f) coef = c;
        }
        out[0] = norm;
        out[1] = coef;
    }
}

struct AdamArgs {
    float lr, beta1, beta2, eps, weight_decay, inv_bc1, inv_bc2;
};

__device__ __forceinline__ void adam_one(float& p, float& m, float& v, float g, const AdamArgs& a) {
    m = a.beta1 * m + (1.0f - a.beta1) * g;
    v = a.beta2 * v + (1.0f - a.beta2) * g * g;
    const float denom = sqrtf(v * a.inv_bc2) + a.eps;
    const float update = (m * a.inv_bc1) / denom + a.weight_decay * p;
    p = p - a.lr * update;
}

// ---- lists of tensors in one launch ----------------------------------------------------------------------------------
// A stack has tens of tensors, most of them small (a norm weight is 3 - 16 KB): one launch per tensor left the update of a
// 63 M parameter stack at 42 launches of which half moved next to nothing.  A list of up to kListMax tensors is cut into
// chunks of kChunk elements, numbered through, that a fixed grid of blocks walks in steps of its size (so the chunks of a
// block, and with them the order of the norm's sums, depend on the list alone).  16 bytes per lane, four vectors of every
// stream in flight per thread.
constexpr int kListMax = 48;
constexpr int kChunk = 4096;             // elements: 4 vectors x 4 floats x 256 threads
constexpr int kListBlocks = 2048;        // 8 per CU
constexpr int kNormBlocks = 1024;        // the norm only reads: 4 per CU reach 6.2 - 6.4 TB/s on one tensor, 8 6.0 - 6.2, 2 5.7

struct TensorList {
    float* a[kListMax];                  // fp32: the gradient (norm), or master / moments / gradient (update)
    float* m[kListMax];
    float* v[kListMax];
    const float* g[kListMax];
    bf16_t* param[kListMax];             // may be null
    int64_t n[kListMax];
    int first[kListMax];                 // launch-wide number of the tensor's first chunk
    int count, chunks;
};

__device__ __forceinline__ int tensor_of(const TensorList& l, int chunk) {  // scalar bisection
    int lo = 0, hi = l.count;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (l.first[mid] <= chunk) lo = mid;
        else hi = mid;
    }
    return lo;
}

__global__ __launch_bounds__(kOptBlock) void sumsq_list_kernel(const TensorList l, float* __restrict__ partials) {
    __shared__ float red[kOptBlock / 64];
    float acc = 0.f;
    for (int chunk = blockIdx.x; chunk < l.chunks; chunk += gridDim.x) {
        const int t = tensor_of(l, chunk);
        const float* g = l.g[t];
        const int64_t base = (int64_t)(chunk - l.first[t]) * kChunk, left = l.n[t] - base;
        if (left >= kChunk) {
            f32x4 x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const f32x4*>(g + base + (u * kOptBlock + threadIdx.x) * 4);
#pragma unroll
            for (int u = 0; u < 4; ++u) acc += x[u][0] * x[u][0] + x[u][1] * x[u][1] + x[u][2] * x[u][2] + x[u][3] * x[u][3];
        } else {
            for (int64_t i = threadIdx.x; i < left; i += kOptBlock) acc += g[base + i] * g[base + i];
        }
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < kOptBlock / 64; ++k) t += red[k];
        partials[blockIdx.x] = t;
    }
}

// The state is touched once per step and is far larger than the last-level cache: streaming loads and stores.
__device__ __forceinline__ f32x4 ld_stream(const float* p, int i) { return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p) + i); }
__device__ __forceinline__ void st_stream(float* p, int i, f32x4 x) { __builtin_nontemporal_store(x, reinterpret_cast<f32x4*>(p) + i); }

// Bound by HBM: 30 B per parameter, 4 more for the norm.  465 M parameters, norm + update: 3.39 - 3.51 ms with one launch per tensor
// and two vectors in flight per stream, 3.15 with this, 3.13 - 3.10 with the streaming hint (5.1 TB/s: the update 2.75 ms, the norm
// 0.37); a training iteration of 63 M parameters 3.06 -> 2.96 ms by the hint.  1024 or 4096 blocks are no different.
// The chunks of a list are walked from the last to the first: the norm, which went through the gradients in the other direction, has left the last
// ones in the last-level cache.  Lists go out first to last, so that with more than kListMax tensors the update begins where nothing is cached
// any more.  465 M parameters, norm + update, with the norm's 1024 instead of 2048 blocks: in 40 tensors 3105 -> 3087 us, in 100 3025 -> 3012.
__global__ __launch_bounds__(kOptBlock) void adamw_list_kernel(const TensorList l, const AdamArgs a, const float* __restrict__ norm_coef) {
    const float coef = norm_coef ? norm_coef[1] : 1.0f;
    for (int chunk = l.chunks - 1 - (int)blockIdx.x; chunk >= 0; chunk -= gridDim.x) {
        const int t = tensor_of(l, chunk);
        const int64_t base = (int64_t)(chunk - l.first[t]) * kChunk, left = l.n[t] - base;
        float *pp = l.a[t] + base, *pm = l.m[t] + base, *pv = l.v[t] + base;
        const float* pg = l.g[t] + base;
        bf16_t* pw = l.param[t] ? l.param[t] + base : nullptr;
        if (left >= kChunk) {
            f32x4 p[4], m[4], v[4], g[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = u * kOptBlock + threadIdx.x;
                p[u] = ld_stream(pp, i); m[u] = ld_stream(pm, i); v[u] = ld_stream(pv, i); g[u] = ld_stream(pg, i);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = u * kOptBlock + threadIdx.x;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float pk = p[u][k], mk = m[u][k], vk = v[u][k];
                    adam_one(pk, mk, vk, g[u][k] * coef, a);
                    p[u][k] = pk; m[u][k] = mk; v[u][k] = vk;
                }
                st_stream(pp, i, p[u]); st_stream(pm, i, m[u]); st_stream(pv, i, v[u]);
                if (pw) {
                    bf16x4 o;
#pragma unroll
                    for (int k = 0; k < 4; ++k) o[k] = (bf16_t)p[u][k];
                    reinterpret_cast<bf16x4*>(pw)[i] = o;
                }
            }
        } else {
            for (int64_t i = threadIdx.x; i < left; i += kOptBlock) {
                float p = pp[i], m = pm[i], v = pv[i];
                adam_one(p, m, v, pg[i] * coef, a);
                pp[i] = p; pm[i] = m; pv[i] = v;
                if (pw) pw[i] = (bf16_t)p;
            }
        }
    }
}

AdamArgs adam_args(float lr, float beta1, float beta2, float eps, float weight_decay, int64_t step, int bias_correction) {
    AdamArgs a;
    a.lr = lr; a.beta1 = beta1; a.beta2 = beta2; a.eps = eps; a.weight_decay = weight_decay;
    a.inv_bc1 = bias_correction ? (float)(1.0 / (1.0 - pow((double)beta1, (double)step))) : 1.0f;
    a.inv_bc2 = bias_correction ? (float)(1.0 / (1.0 - pow((double)beta2, (double)step))) : 1.0f;
    return a;
}

// Whether an update of the list writes memory that tensor `slot` is made of: a parameter that occurs twice is updated twice, one
// launch after the other.
bool updates_meet(const TensorList& l, int slot) {
    auto meet = [&](const void* const* streams, int size) {
        const char* p = (const char*)streams[slot];
        for (int i = 0; i < slot && p; ++i) {
            const char* q = (const char*)streams[i];
            if (q && p < q + l.n[i] * size && q < p + l.n[slot] * size) return true;
        }
        return false;
    };
    return meet((const void* const*)l.a, 4) || meet((const void* const*)l.m, 4) || meet((const void* const*)l.v, 4) ||
           meet((const void* const*)l.param, 2);
}

// calls launch(list, number of blocks) for every kListMax non-empty tensors of 0 .. count - 1, and earlier in front of a tensor
// that must_wait(list, slot); fill(list, slot, i) sets the pointers
template <class Fill, class Wait, class Launch>
void for_each_list(int count, const int64_t* n, Fill fill, Wait must_wait, Launch launch) {
    TensorList l;
    l.count = l.chunks = 0;
    auto flush = [&]() {
        if (l.count) launch(l, (unsigned)(l.chunks < kListBlocks ? l.chunks : kListBlocks));
        l.count = l.chunks = 0;
    };
    for (int i = 0; i < count; ++i) {
        if (n[i] == 0) continue;
        const int64_t chunks = (n[i] + kChunk - 1) / kChunk;
        if (l.count == kListMax || l.chunks + chunks >= (1LL << 30)) flush();
        fill(l, l.count, i);
        l.n[l.count] = n[i];
        if (must_wait(l, l.count)) {
            flush();
            fill(l, 0, i);
            l.n[0] = n[i];
        }
        l.first[l.count] = l.chunks;
        l.chunks += (int)chunks;
        ++l.count;
    }
    flush();
}

}  // namespace

extern "C" int64_t ezl_sumsq_partials(void) { return kSumsqPartials; }

extern "C" int ezl_sumsq_f32(const void* x, int64_t n, void* partials, void* stream) {
    EZL_REQUIRE(n >= 0 && partials && (n == 0 || x), EZL_EINVAL, "ezl_sumsq_f32: null pointer");
    EZL_REQUIRE(ezl_aligned16(x), EZL_EINVAL, "ezl_sumsq_f32: x must be 16-byte aligned");
    // always kSumsqPartials blocks, so every slot of `partials` is written (zeros for blocks without work)
    hipLaunchKernelGGL(sumsq_partial_kernel, dim3(kSumsqPartials), dim3(kSumsqBlock), 0, (hipStream_t)stream, (const float*)x, n,
                       (float*)partials);
    EZL_LAUNCH_CHECK("ezl_sumsq_f32");
    return EZL_OK;
}

extern "C" int ezl_clip_coef(const void* partials, int64_t count, float max_norm, void* norm_coef_out, void* stream) {
    EZL_REQUIRE(count >= 0 && norm_coef_out && (count == 0 || partials), EZL_EINVAL, "ezl_clip_coef: null pointer");
    hipLaunchKernelGGL(clip_coef_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, (const float*)partials, count, max_norm,
                       (float*)norm_coef_out);
    EZL_LAUNCH_CHECK("ezl_clip_coef");
    return EZL_OK;
}

extern "C" int ezl_adamw_step(void* master, void* exp_avg, void* exp_avg_sq, const void* grad, void* param_bf16, int64_t n,
                              float lr, float beta1, float beta2, float eps, float weight_decay, int64_t step,
                              int bias_correction, const void* norm_coef, void* stream) {
    EZL_REQUIRE(n >= 0 && (n == 0 || (master && exp_avg && exp_avg_sq && grad)), EZL_EINVAL, "ezl_adamw_step: null pointer");
    EZL_REQUIRE(step >= 1, EZL_EINVAL, "ezl_adamw_step: step counts from 1");
    EZL_REQUIRE(ezl_aligned16(master) && ezl_aligned16(exp_avg) && ezl_aligned16(exp_avg_sq) && ezl_aligned16(grad) &&
                    (((uintptr_t)param_bf16 & 7) == 0),
                EZL_EINVAL, "ezl_adamw_step: fp32 buffers must be 16-byte aligned, the bf16 weight 8-byte aligned");
    const int64_t one[1] = {n};
    const AdamArgs a = adam_args(lr, beta1, beta2, eps, weight_decay, step, bias_correction);
    for_each_list(1, one, [&](TensorList& l, int s, int) {
        l.a[s] = (float*)master; l.m[s] = (float*)exp_avg; l.v[s] = (float*)exp_avg_sq; l.g[s] = (const float*)grad; l.param[s] = (bf16_t*)param_bf16;
    }, updates_meet, [&](const TensorList& l, unsigned blocks) {
        hipLaunchKernelGGL(adamw_list_kernel, dim3(blocks), dim3(kOptBlock), 0, (hipStream_t)stream, l, a, (const float*)norm_coef);
    });
    EZL_LAUNCH_CHECK("ezl_adamw_step");
    return EZL_OK;
}

// fp32 slots that ezl_sumsq_list fills for a list of `count` tensors
extern "C" int64_t ezl_sumsq_list_partials(int count) { return count < 0 ? -1 : ((int64_t)count + kListMax - 1) / kListMax * kNormBlocks; }

extern "C" int ezl_sumsq_list(int count, const void* const* x, const int64_t* n, void* partials, void* stream) {
    EZL_REQUIRE(count >= 0 && (count == 0 || (x && n && partials)), EZL_EINVAL, "ezl_sumsq_list: bad count or null argument array");
    for (int i = 0; i < count; ++i)
        EZL_REQUIRE(n[i] >= 0 && n[i] < (1LL << 40) && (n[i] == 0 || x[i]) && ezl_aligned16(x[i]), EZL_EINVAL,
                    "ezl_sumsq_list: null or misaligned tensor");
    float* out = (float*)partials;
    float* const end = out + ezl_sumsq_list_partials(count);
    for_each_list(count, n, [&](TensorList& l, int s, int i) { l.g[s] = (const float*)x[i]; }, [](const TensorList&, int) { return false; },
                  [&](const TensorList& l, unsigned blocks) {
        if (blocks > kNormBlocks) blocks = kNormBlocks;
        hipLaunchKernelGGL(sumsq_list_kernel, dim3(blocks), dim3(kOptBlock), 0, (hipStream_t)stream, l, out);
        out += blocks;
    });
    if (out < end)  // slots of blocks that were not needed (a fill kernel, not a memset node)
        hipLaunchKernelGGL(zero_f32_kernel, dim3((unsigned)((end - out + 255) / 256)), dim3(256), 0, (hipStream_t)stream, out, (int)(end - out));
    EZL_LAUNCH_CHECK("ezl_sumsq_list");
    return EZL_OK;
}

extern "C" int ezl_adamw_list(int count, void* const* master, void* const* exp_avg, void* const* exp_avg_sq, const void* const* grad,
                              void* const* param_bf16, const int64_t* n, float lr, float beta1, float beta2, float eps, float weight_decay,
                              int64_t step, int bias_correction, const void* norm_coef, void* stream) {
    EZL_REQUIRE(count >= 0 && (count == 0 || (master && exp_avg && exp_avg_sq && grad && param_bf16 && n)), EZL_EINVAL,
                "ezl_adamw_list: bad count or null argument array");
    EZL_REQUIRE(step >= 1, EZL_EINVAL, "ezl_adamw_list: step counts from 1");
    for (int i = 0; i < count; ++i) {
        EZL_REQUIRE(n[i] >= 0 && n[i] < (1LL << 40) && (n[i] == 0 || (master[i] && exp_avg[i] && exp_avg_sq[i] && grad[i])), EZL_EINVAL,
                    "ezl_adamw_list: null pointer");
        EZL_REQUIRE(ezl_aligned16(master[i]) && ezl_aligned16(exp_avg[i]) && ezl_aligned16(exp_avg_sq[i]) && ezl_aligned16(grad[i]) &&
                        (((uintptr_t)param_bf16[i] & 7) == 0),
                    EZL_EINVAL, "ezl_adamw_list: fp32 buffers must be 16-byte aligned, the bf16 weight 8-byte aligned");
    }
    const AdamArgs a = adam_args(lr, beta1, beta2, eps, weight_decay, step, bias_correction);
    for_each_list(count, n, [&](TensorList& l, int s, int i) {
        l.a[s] = (float*)master[i]; l.m[s] = (float*)exp_avg[i]; l.v[s] = (float*)exp_avg_sq[i]; l.g[s] = (const float*)grad[i];
        l.param[s] = (bf16_t*)param_bf16[i];
    }, updates_meet, [&](const TensorList& l, unsigned blocks) {
        hipLaunchKernelGGL(adamw_list_kernel, dim3(blocks), dim3(kOptBlock), 0, (hipStream_t)stream, l, a, (const float*)norm_coef);
    });
    EZL_LAUNCH_CHECK("ezl_adamw_list");
    return EZL_OK;
}
