// HBM-bound elementwise / gather kernels of the llama decoder-layer step (gfx950):
// SwiGLU, rotary embedding, token-embedding gather / scatter-add, [b,s,h] <-> [s,b,h] row moves,
// bf16 add and bf16 <-> fp32 casts.  All use 128-bit accesses (8 bf16 per lane).
#include "common.h"
#include "qkv_bias.h"

#include <type_traits>

namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(int64_t items, int per_block, int64_t cap = 256 * 32) {
    int64_t g = (items + per_block - 1) / per_block;
    if (g > cap) g = cap;
    if (g < 1) g = 1;
    return (unsigned)g;
}

// 1 / (1 + 2^(-x log2 e)) with the bare exp2 / rcp instructions (1 ulp each); saturates correctly at both ends
__device__ __forceinline__ float sigmoidf_fast(float x) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f));
}

// ---------------------------------------------------------------------------------------------
// SwiGLU: out = silu(gate) * up     (llama/transformer.py:220-222, glu_activations.py:56-61)
// ---------------------------------------------------------------------------------------------
// STREAM: results past the caches (ezl_streams).  Where one of them fits it is read next by products whose operands every XCD fetches for itself: input
// gradient over gate and up behind the backward kernel, 1531 x 4096 x 22016, 349 -> 303 us with plain stores; a layer's forward and backward over
// 1531 tokens at h = 4096 687 -> 672 and 1535 -> 1483 us, over 4096 tokens 1511 -> 1490 and 3339 -> 3325.
template <bool STREAM>
__global__ __launch_bounds__(kBlock) void swiglu_fwd_kernel(const bf16_t* __restrict__ gate, const bf16_t* __restrict__ up,
                                                            bf16_t* __restrict__ out, int64_t n8) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += (int64_t)gridDim.x * kBlock) {
        float g[8], u[8], o[8];
        unpack8(ld_bf16x8_nt(gate + i * 8), g);
        unpack8(ld_bf16x8_nt(up + i * 8), u);
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = g[k] * sigmoidf_fast(g[k]) * u[k];
        st_result<STREAM>(out + i * 8, pack8(o));
    }
}

// dgate = dout * up * s * (1 + g * (1 - s)),  dup = dout * g * s,  s = sigmoid(g)
template <bool STREAM>
__global__ __launch_bounds__(kBlock) void swiglu_bwd_kernel(const bf16_t* __restrict__ dout, const bf16_t* __restrict__ gate,
                                                            const bf16_t* __restrict__ up, bf16_t* __restrict__ dgate,
                                                            bf16_t* __restrict__ dup, int64_t n8) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += (int64_t)gridDim.x * kBlock) {
        float g[8], u[8], d[8], dg[8], du[8];
        unpack8(ld_bf16x8_nt(gate + i * 8), g);
        unpack8(ld_bf16x8_nt(up + i * 8), u);
        unpack8(ld_bf16x8_nt(dout + i * 8), d);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float s = sigmoidf_fast(g[k]);
            dg[k] = d[k] * u[k] * s * (1.0f + g[k] * (1.0f - s));
            du[k] = d[k] * g[k] * s;
        }
        st_result<STREAM>(dgate + i * 8, pack8(dg));
        st_result<STREAM>(dup + i * 8, pack8(du));
    }
}

// ---------------------------------------------------------------------------------------------
// Rotary embedding (llama/positional_embeddings.py:17-36, 94-96, 105-122)
// ---------------------------------------------------------------------------------------------
// cos/sin table [npos, d/2] in fp32: theta = (p / scale_factor) * inv_freq[j]  (:21-23)
__global__ __launch_bounds__(kBlock) void rope_table_kernel(const float* __restrict__ inv_freq, float* __restrict__ cosb,
                                                            float* __restrict__ sinb, int64_t npos, int half,
                                                            float scale_factor) {
    const int64_t n = npos * half;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const int64_t p = i / half;
        const int j = (int)(i % half);
        const float t = (float)p / scale_factor;
        const float th = t * inv_freq[j];
        cosb[i] = cosf(th);
        sinb[i] = sinf(th);
    }
}

// x [rows = s*b (s-major), nheads, d] with a row stride; one work item = 8 low-half + 8 high-half
// elements of one head.  out1 = x1*c - sign*x2*s ; out2 = x2*c + sign*x1*s  (sign = -1: backward).
// Two tensors that share their rows (q and k of one layer: nheads0 + nheads1 heads per row) go through one launch; the
// second is absent when nheads1 == 0.
struct RopeSide {
    const bf16_t* x;
    bf16_t* out;
    int64_t in_stride, out_stride;
};

__global__ __launch_bounds__(kBlock) void rope_kernel(RopeSide a, RopeSide b2, const float* __restrict__ cosb,
                                                      const float* __restrict__ sinb, const int64_t* __restrict__ position_ids,
                                                      int64_t rows, int s, int b, int nheads0, int nheads1, int d, int64_t npos,
                                                      float sign) {
    const int half = d >> 1;
    const int per_head = half >> 3;
    const int nheads = nheads0 + nheads1;
    const int64_t items = rows * nheads * per_head;
    for (int64_t it = (int64_t)blockIdx.x * kBlock + threadIdx.x; it < items; it += (int64_t)gridDim.x * kBlock) {
        const int j8 = (int)(it % per_head);
        const int64_t rh = it / per_head;
        int head = (int)(rh % nheads);
        const int64_t row = rh / nheads;
        const int si = (int)(row / b), bi = (int)(row % b);
        int64_t pos = position_ids ? position_ids[(int64_t)bi * s + si] : si;
        pos = pos < 0 ? 0 : (pos >= npos ? npos - 1 : pos);
        const float* cp = cosb + pos * half + j8 * 8;
        const float* sp = sinb + pos * half + j8 * 8;
        const bool second = head >= nheads0;
        head -= second ? nheads0 : 0;
        const bf16_t* xi = (second ? b2.x : a.x) + row * (second ? b2.in_stride : a.in_stride) + (int64_t)head * d + j8 * 8;
        bf16_t* xo = (second ? b2.out : a.out) + row * (second ? b2.out_stride : a.out_stride) + (int64_t)head * d + j8 * 8;
        float av[8], c[8], o1[8], o2[8];
        unpack8(ld_bf16x8(xi), av);
        unpack8(ld_bf16x8(xi + half), c);
        const f32x4 c0 = *reinterpret_cast<const f32x4*>(cp), c1 = *reinterpret_cast<const f32x4*>(cp + 4);
        const f32x4 s0 = *reinterpret_cast<const f32x4*>(sp), s1 = *reinterpret_cast<const f32x4*>(sp + 4);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float cs = k < 4 ? c0[k] : c1[k - 4];
            const float sn = sign * (k < 4 ? s0[k] : s1[k - 4]);
            o1[k] = av[k] * cs - c[k] * sn;
            o2[k] = c[k] * cs + av[k] * sn;
        }
        st_bf16x8(xo, pack8(o1));
        st_bf16x8(xo + half, pack8(o2));
    }
}

// ---------------------------------------------------------------------------------------------
// Token embedding (base_modules/layers/vocab_parallel_emb.py:106-137, TP=1)
// ---------------------------------------------------------------------------------------------
// What a range test found, 1 for an id >= limit and 2 for a negative one: ORed into a word of device memory, or, HOST, byte 0 and
// byte 1 of pinned host memory set by plain stores.  Those need neither a clearing launch before the kernel nor a copy behind it,
// which cost a host-bound step 8 us of host time and the GPU a copy-engine hand-over; an atomic OR on host memory is not among
// those that PCIe carries.
template <bool HOST>
__device__ __forceinline__ void raise_id_flag(void* flag, int bad) {
    if constexpr (HOST) {
        if (bad & 1) ((volatile unsigned char*)flag)[0] = 1;
        if (bad & 2) ((volatile unsigned char*)flag)[1] = 1;
    } else if (bad) {
        atomicOr((int*)flag, bad);
    }
}

// the range test of an index tensor, without a host sync
template <bool HOST>
__global__ __launch_bounds__(kBlock) void ids_in_range_kernel(const int64_t* __restrict__ ids, int64_t n, int64_t limit, void* bad_flag) {
    int bad = 0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const int64_t id = ids[i];
        bad |= id >= limit ? 1 : (id < 0 ? 2 : 0);
    }
    raise_id_flag<HOST>(bad_flag, bad);
}

// out[r, :] = W[ids[r], :]; an id outside [0, V) raises the flag and yields a zero row.
// One wave per row; a lane's loads (up to 8 vectors of 8 at a time: a row of 4096 in one go) are all in flight before its
// first store.
template <bool HOST>
__global__ __launch_bounds__(kBlock) void embed_gather_kernel(const int64_t* __restrict__ ids, const bf16_t* __restrict__ W,
                                                              bf16_t* __restrict__ out, int64_t rows, int h, int64_t V, void* bad_flag,
                                                              const RowSwap swap) {
    const int h8 = h >> 3;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int64_t r = (int64_t)blockIdx.x * 4 + wave; r < rows; r += (int64_t)gridDim.x * 4) {
        const int64_t id = ids[r];
        const bool ok = id >= 0 && id < V;
        if (!ok && lane == 0) raise_id_flag<HOST>(bad_flag, id >= V ? 1 : 2);
        const bf16_t* src = W + (ok ? id : 0) * h;
        bf16_t* dst = out + (swap.d1 ? (int64_t)swapped_row((int)r, swap) : r) * h;
        for (int c0 = lane; c0 < h8; c0 += 512) {
            bf16x8 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
#pragma unroll
                for (int k = 0; k < 8; ++k) v[u][k] = (bf16_t)0.0f;
                if (ok && c0 + u * 64 < h8) v[u] = ld_bf16x8(src + (c0 + u * 64) * 8);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (c0 + u * 64 < h8) st_bf16x8(dst + (c0 + u * 64) * 8, v[u]);
        }
    }
}

// dW[id, :] += sum of dY[r, :] over all rows r with ids[r] == id, in increasing row order (bit-reproducible), in time
// linear in the number of rows.  The rows are bucketed by id through four int32 tables in the workspace:
//   cnt[V]   rows per id                      first[V]  smallest row holding the id (its block does the sum)
//   off[V]   start of the id's bucket         bucket[T] rows grouped by id (order inside a group: as the atomics fell)
// The owner block of an id sorts that id's bucket by row number before summing, so the order the atomics produced never
// reaches the result.  Ids with more than kOwnedRows rows (a padding token, frequent words) are left to several blocks each,
// a slice of the columns per block.
constexpr int kOwnedRows = 32;
inline int64_t embed_heavy_max(int64_t rows) { return rows / kOwnedRows + 1; }  // more ids than this cannot be that frequent

// The lanes of the wave that hold the same id as its first active lane (a run of padding is all of them), and whether this lane
// is one of them: their atomics on one address become one.
__device__ __forceinline__ bool same_as_first_lane(int id, unsigned long long& mask) {
    const bool same = id == __builtin_amdgcn_readfirstlane(id);
    mask = __ballot(same);
    return same;
}

__global__ __launch_bounds__(kBlock) void embed_tables_init_kernel(int* __restrict__ cnt, int* __restrict__ first,
                                                                   int* __restrict__ fill, int* __restrict__ cursor, int64_t V) {
    if (blockIdx.x == 0 && threadIdx.x < 2) cursor[threadIdx.x] = 0;  // next free bucket entry, number of frequent ids
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < V; i += (int64_t)gridDim.x * kBlock) {
        cnt[i] = 0;
        fill[i] = 0;
        first[i] = 0x7fffffff;
    }
}

__global__ __launch_bounds__(kBlock) void embed_count_kernel(const int64_t* __restrict__ ids, int* __restrict__ cnt,
                                                             int* __restrict__ first, int64_t rows, int64_t V) {
    for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < rows; r += (int64_t)gridDim.x * kBlock) {
        const int64_t id = ids[r];
        if (id < 0 || id >= V) continue;
        unsigned long long mask;
        if (!same_as_first_lane((int)id, mask)) {
            atomicAdd(cnt + id, 1);
            atomicMin(first + id, (int)r);
        } else if ((int)(threadIdx.x & 63) == __builtin_ctzll(mask)) {  // the lowest lane holds the smallest row
            atomicAdd(cnt + id, (int)__popcll(mask));
            atomicMin(first + id, (int)r);
        }
    }
}

// off[id] = start of id's range in the bucket array.  The ranges only have to be disjoint -- every bucket is put into row
// order before it is summed, and where it lies does not reach the result -- so the owner row of each id (its smallest row)
// takes the next cnt[id] entries from a running cursor; no prefix sum over the vocabulary is needed.
__global__ __launch_bounds__(kBlock) void embed_assign_kernel(const int64_t* __restrict__ ids, const int* __restrict__ cnt,
                                                              const int* __restrict__ first, int* __restrict__ off,
                                                              int* __restrict__ cursor, int* __restrict__ heavy, int64_t rows,
                                                              int64_t V) {
    for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < rows; r += (int64_t)gridDim.x * kBlock) {
        const int64_t id = ids[r];
        if (id < 0 || id >= V || first[id] != (int)r) continue;
        const int n = cnt[id];
        off[id] = atomicAdd(cursor, n);
        if (n > kOwnedRows) heavy[atomicAdd(cursor + 1, 1)] = (int)id;
    }
}

__global__ __launch_bounds__(kBlock) void embed_bucket_kernel(const int64_t* __restrict__ ids, const int* __restrict__ off,
                                                              int* __restrict__ fill, int* __restrict__ bucket, int64_t rows,
                                                              int64_t V) {
    for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < rows; r += (int64_t)gridDim.x * kBlock) {
        const int64_t id = ids[r];
        if (id < 0 || id >= V) continue;
        unsigned long long mask;
        int at;
        if (!same_as_first_lane((int)id, mask)) {
            at = atomicAdd(fill + id, 1);
        } else {
            const int lane = threadIdx.x & 63, leader = __builtin_ctzll(mask);
            int base = 0;
            if (lane == leader) base = atomicAdd(fill + id, (int)__popcll(mask));
            at = __builtin_amdgcn_readlane(base, leader) + (int)__popcll(mask & ((1ull << lane) - 1));
        }
        bucket[off[id] + at] = (int)r;
    }
}

// The four kernels above as one workgroup, for short batches: each of those launches costs more than its work there.  Ids are looked up in a hash
// table in LDS, so the global tables are only written: cnt / first / off of the ids that occur, and, with zero_all, cnt = 0 of all others.
// Bound by LDS atomics, hence by the rows (and with zero_all by one workgroup's stores, hence by the vocabulary).  The whole gradient, h = 256, us,
// four launches against this, adding / overwriting; ids drawn evenly, as frequent as words (1 / rank), all the same (padding):
//   V = 32000    512 rows 16.2 / 23.3, 9.6 / 17.9; 18.3 / 22.7, 11.4 / 16.8; 26.6 / 28.3, 20.5 / 23.1
//               1531      17.0 / 23.8, 13.3 / 21.3; 21.5 / 24.1, 16.0 / 19.9; 51.1 / 52.5, 45.1 / 47.5
//               2048      17.9 / 24.1, 17.4 / 25.1; 25.1 / 27.6, 21.6 / 24.7; 63.0 / 64.4, 56.9 / 59.0
//               4096      20.0 / 25.6, 27.7 / 34.4; 29.1 / 30.9, 29.1 / 31.6; 114 / 116, 109 / 110
//   V = 131072  1531      17.0 / 43.1, 13.5 / 41.9; 21.2 / 44.5, 15.7 / 39.9
//               2048      17.4 / 42.2, 17.0 / 45.2; 22.0 / 42.4, 18.0 / 41.5
// (Without the lanes of a wave that hold one id sharing their atomics 2048 equal ids took 62.5 / 65.1.)
constexpr int kSmallRows = 2048, kSmallRowsZero = 1536, kSmallSlots = 2 * kSmallRows, kSmallThreads = 1024;
constexpr int64_t kSmallVocab = 131072;  // with zero_all
__global__ __launch_bounds__(kSmallThreads) void embed_tables_small_kernel(const int64_t* __restrict__ ids, int* __restrict__ cnt, int* __restrict__ first,
                                                                           int* __restrict__ off, int* __restrict__ bucket, int* __restrict__ cursor,
                                                                           int* __restrict__ heavy, int rows, int64_t V, int zero_all) {
    __shared__ int s_id[kSmallSlots], s_cnt[kSmallSlots], s_first[kSmallSlots], s_off[kSmallSlots];
    __shared__ int s_next, s_heavy;
    constexpr int PER = kSmallRows / kSmallThreads;
    const int tid = threadIdx.x, lane = tid & 63;
    int row_id[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int r = k * kSmallThreads + tid;
        const int64_t id = r < rows ? ids[r] : -1;
        row_id[k] = id >= 0 && id < V ? (int)id : -1;
    }
    // (2048 or 4096 slots, the hash's highest bits: at most half of them are ever taken)
    const int shift = rows <= kSmallRows / 4 ? 21 : 20, slots = 1 << (32 - shift);
    for (int i = tid; i < slots; i += kSmallThreads) {
        s_id[i] = -1;
        s_cnt[i] = 0;
        s_first[i] = 0x7fffffff;
    }
    if (tid == 0) s_next = s_heavy = 0;
    if (zero_all)
        for (int64_t i = tid; i < V; i += kSmallThreads) cnt[i] = 0;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the zeros have arrived before the counts below are stored
    __syncthreads();
    int slot[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int r = k * kSmallThreads + tid;
        slot[k] = -1;
        const int id = row_id[k];
        if (id < 0) continue;
        unsigned long long mask;
        const bool same = same_as_first_lane(id, mask);
        const int leader = __builtin_ctzll(mask);
        if (!same || lane == leader) {
            unsigned i = ((unsigned)id * 0x9E3779B1u) >> shift;
            for (;;) {  // ends: half of the slots stay free
                const int old = atomicCAS(&s_id[i], -1, id);
                if (old == -1 || old == id) break;
                i = (i + 1) & (slots - 1);
            }
            slot[k] = (int)i;
            atomicAdd(&s_cnt[i], same ? (int)__popcll(mask) : 1);
            atomicMin(&s_first[i], r);  // (the lowest lane holds the smallest row)
        }
        const int shared = __builtin_amdgcn_readlane(slot[k], leader);
        if (same) slot[k] = shared;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int r = k * kSmallThreads + tid;
        if (slot[k] < 0 || s_first[slot[k]] != r) continue;
        const int id = s_id[slot[k]], n = s_cnt[slot[k]], o = atomicAdd(&s_next, n);
        s_off[slot[k]] = o;
        cnt[id] = n;
        first[id] = r;
        off[id] = o;
        if (n > kOwnedRows) heavy[atomicAdd(&s_heavy, 1)] = id;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        if (slot[k] < 0) continue;
        unsigned long long mask;
        const bool same = same_as_first_lane(slot[k], mask);
        const int leader = __builtin_ctzll(mask);
        int at = 0;
        if (!same || lane == leader) at = atomicAdd(&s_off[slot[k]], same ? (int)__popcll(mask) : 1);
        const int base = __builtin_amdgcn_readlane(at, leader);
        if (same) at = base + (int)__popcll(mask & ((1ull << lane) - 1));
        bucket[at] = k * kSmallThreads + tid;
    }
    if (tid == 0) cursor[1] = s_heavy;
}
static_assert(kSmallSlots == 1 << (32 - 20), "the largest table");

// p[0 .. n4) = 0 in 16-byte pieces: a block clears one contiguous 16 KiB chunk (4 stores per thread), chunks dealt to blocks in
// order, so the blocks running at any moment sweep one window of the buffer.
__global__ __launch_bounds__(kBlock) void zero_f32x4_kernel(f32x4* __restrict__ p, int64_t n4) {
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    for (int64_t c = blockIdx.x; c * (4 * kBlock) < n4; c += gridDim.x) {
        const int64_t i0 = c * (4 * kBlock) + threadIdx.x;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i0 + u * kBlock < n4) p[i0 + u * kBlock] = z;
    }
}

// What putting the rows of a frequent id in order needs of LDS.
constexpr int kListRows = 2048;               // rows in order at a time
constexpr int kWindowWords = 2048;            // words of the bitmap over row numbers
constexpr int kWindowRows = 32 * kWindowWords;
constexpr int kFrequentBlocks = 1024;         // 512: each of 3971 ids 33 times, h = 4096, 448 us instead of 341
struct EmbedOrder {
    alignas(16) int list[kListRows];
    int raw[kBlock];
    unsigned bits[kWindowWords];
    int wave_total[kBlock / 64];
};

// One frequent id, columns col0 + 2 thread, + 1: a thread walks the id's rows in order with up to 24 rows' loads in flight (one
// register each), so that the time is the latency of n / 24 loads rather than of n / 4.  (1000 padding rows of 4000, h = 2048:
// the scatter kernel 430 -> 79 us.)
// Every slice of the columns puts the rows in order for itself, which must not cost more than adding them: up to one row per thread
// by rank, whatever the batch; more through a bitmap over 65536 row numbers at a time.  The whole gradient, added to a buffer, of
// T rows of 4096 by one block per id, by column slices over bitmap windows of 2048 rows, and so: T = 131072, each id 33 times
// 334, 3473, 340 us; 300 times 474, 1043, 310; 3000 times 3335, 922, 636; T = 16384, ids by Zipf's law 950, 164, 148.
template <typename OutT>
__device__ __forceinline__ void embed_frequent_id(const bf16_t* __restrict__ dY, OutT* __restrict__ dW, const int* __restrict__ mine, int n,
                                                  int64_t id, int col0, int64_t rows, int h, int overwrite, EmbedOrder& o, const RowSwap& swap) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int col = col0 + 2 * tid;
    const bool live = col < h;
    const int lane_col = live ? col : 0;
    float a0 = 0.f, a1 = 0.f;
    for (int64_t w0 = 0; w0 < rows; w0 += n <= kBlock ? rows : kWindowRows) {
        __syncthreads();  // the previous window's (or id's) LDS use is over
        int m = 0;  // rows of the window
        // a thread owns `per` consecutive words of the bitmap; their bits, counted and scanned over the block, say where its rows go
        const int words = rows - w0 < kWindowRows ? (int)((rows - w0 + 31) >> 5) : kWindowWords, per = (words + kBlock - 1) / kBlock;
        const int last = (tid + 1) * per < words ? (tid + 1) * per : words;
        if (n <= kBlock) {  // rows are distinct: rank = number of smaller rows
            const int v = tid < n ? mine[tid] : 0x7fffffff;
            o.raw[tid] = v;
            __syncthreads();
            int rank = 0;
            for (int j = 0; j < n; ++j) rank += o.raw[j] < v;
            if (tid < n) o.list[rank] = swapped_row(v, swap);
            m = n;
        } else {
            for (int i = tid; i < words; i += kBlock) o.bits[i] = 0u;
            __syncthreads();
            for (int i = tid; i < n; i += kBlock) {
                const int64_t r = (int64_t)mine[i] - w0;
                if (r >= 0 && r < kWindowRows) atomicOr(&o.bits[r >> 5], 1u << (r & 31));
            }
            __syncthreads();
            int count = 0;
            for (int i = tid * per; i < last; ++i) count += __builtin_popcount(o.bits[i]);
            int end = count;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int v = __shfl_up(end, d, 64);
                if (lane >= d) end += v;
            }
            if (lane == 63) o.wave_total[wv] = end;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kBlock / 64; ++i) {
                if (i < wv) end += o.wave_total[i];
                m += o.wave_total[i];
            }
            m = __builtin_amdgcn_readfirstlane(m);
            o.raw[tid] = end - count;  // (not a register each while rows are added)
        }
        for (int at = 0; at < m; at += kListRows) {
            if (at) __syncthreads();  // the rows before these are added
            if (n > kBlock) {
                int q = o.raw[tid] - at;
                for (int i = tid * per; i < last && q < kListRows; ++i) {
                    unsigned w = o.bits[i];
                    if (q + 32 <= 0) {
                        q += __builtin_popcount(w);
                        continue;
                    }
                    for (; w; w &= w - 1, ++q)
                        if (q >= 0 && q < kListRows) o.list[q] = swapped_row((int)w0 + 32 * i + __builtin_ctz(w), swap);
                }
            }
            __syncthreads();
            const int listed = m - at < kListRows ? m - at : kListRows;
            int i = 0;
            auto batch = [&](auto N) {
                constexpr int U = decltype(N)::value;
                for (; i + U <= listed; i += U) {
                    bf16x2 v[U];
                    int at_row[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) at_row[u] = __builtin_amdgcn_readfirstlane(o.list[i + u]);
#pragma unroll
                    for (int u = 0; u < U; ++u)  // (scalar row address + one lane offset: no address registers per row)
                        v[u] = reinterpret_cast<const bf16x2*>(dY + (int64_t)at_row[u] * h)[lane_col >> 1];
                    __builtin_amdgcn_sched_barrier(0);  // (or the loads are waited for one by one to save registers: 1000 rows 264 us)
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        a0 += (float)v[u][0];
                        a1 += (float)v[u][1];
                    }
                }
            };
            batch(std::integral_constant<int, 24>{});
            batch(std::integral_constant<int, 4>{});
            batch(std::integral_constant<int, 1>{});
        }
    }
    if (!live) return;
    if constexpr (sizeof(OutT) == 2) {
        *reinterpret_cast<bf16x2*>(dW + id * h + col) = bf16x2{(bf16_t)a0, (bf16_t)a1};
    } else {
        f32x2* dst = reinterpret_cast<f32x2*>(dW + id * h + col);
        f32x2 o = {a0, a1};
        if (!overwrite) {
            const f32x2 old = *dst;
            o[0] += old[0];
            o[1] += old[1];
        }
        *dst = o;
    }
}

// overwrite: dW[id] = sum instead of dW[id] += sum, and the rows of ids that do not occur are zero-filled (the whole
// [V, h] gradient is then defined by this launch: no separate fill pass).
// (rows of up to 4096: six waves per SIMD, as the zero fill wants them)
// OutT bf16: the fp32 sums are rounded once as they are stored.  A gradient without an fp32 buffer behind it used to be written in
// fp32, read by a cast and written again, five times the bytes of the result.  Gradient
// of [V, h] over T rows, with the cast and now: 50304 x 1024, T 1167 98 -> 33 us; 32000 x 4096, T 4096 263 -> 59; 152064 x 5120
// 1548 -> 304 (5.1 TB/s, on either side of the flat fill's line).
template <int MAXC, typename OutT>
__global__ __launch_bounds__(kBlock, MAXC == 2 ? 6 : 1) void embed_scatter_bucket_kernel(const int64_t* __restrict__ ids, const bf16_t* __restrict__ dY,
                                                                      OutT* __restrict__ dW, const int* __restrict__ cnt,
                                                                      const int* __restrict__ first, const int* __restrict__ off,
                                                                      const int* __restrict__ bucket, const int* __restrict__ cursor,
                                                                      const int* __restrict__ heavy, int64_t rows, int h, int64_t V,
                                                                      int overwrite, const RowSwap swap) {
    __shared__ EmbedOrder order;
    int *const raw = order.raw, *const sorted = order.list;  // rows of the current id as they are found, and in increasing order
    const int h8 = h >> 3;
    const int helpers = (int)gridDim.x < kFrequentBlocks ? (int)gridDim.x : kFrequentBlocks;
    if ((int)blockIdx.x < helpers) {  // the frequent ids first, as they take longest; the other blocks need not even look
        const int slices = (h + 2 * kBlock - 1) / (2 * kBlock), items = cursor[1] * slices;
        for (int it = blockIdx.x; it < items; it += helpers) {
            const int id = heavy[it / slices];
            embed_frequent_id(dY, dW, bucket + off[id], cnt[id], id, (it % slices) * 2 * kBlock, rows, h, overwrite, order, swap);
        }
        __syncthreads();
    }
    for (int64_t t = blockIdx.x; t < rows; t += gridDim.x) {
        const int64_t id = ids[t];
        if (id < 0 || id >= V) continue;
        if (first[id] != (int)t) continue;  // the block of the smallest row of an id owns it (uniform over the block)
        const int n = cnt[id];
        if (n > kOwnedRows) continue;
        const int* mine = bucket + off[id];
        float acc[MAXC][8];
#pragma unroll
        for (int c = 0; c < MAXC; ++c)
#pragma unroll
            for (int k = 0; k < 8; ++k) acc[c][k] = 0.f;
        auto add_row = [&](int64_t jj) {
#pragma unroll
            for (int c = 0; c < MAXC; ++c) {
                const int col = (c * kBlock + threadIdx.x);
                if (col < h8) {
                    float g[8];
                    unpack8(ld_bf16x8(dY + jj * h + col * 8), g);
#pragma unroll
                    for (int k = 0; k < 8; ++k) acc[c][k] += g[k];
                }
            }
        };
        // rows lst[0 .. m-1] in that order, the loads of four rows in flight at a time
        auto add_rows = [&](const int* lst, int m) {
            int i = 0;
            for (; i + 4 <= m; i += 4) {
                bf16x8 v[4][MAXC];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int64_t jj = lst[i + u];
#pragma unroll
                    for (int c = 0; c < MAXC; ++c) {
                        const int col = (c * kBlock + threadIdx.x);
                        if (col < h8) v[u][c] = ld_bf16x8(dY + jj * h + col * 8);
                    }
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int c = 0; c < MAXC; ++c) {
                        const int col = (c * kBlock + threadIdx.x);
                        if (col < h8) {
#pragma unroll
                            for (int k = 0; k < 8; ++k) acc[c][k] += (float)v[u][c][k];
                        }
                    }
            }
            for (; i < m; ++i) add_row(lst[i]);
        };
        if (n == 1) {
            add_row(swapped_row((int)t, swap));
        } else {
            __syncthreads();  // the previous id's LDS use is over
            if ((int)threadIdx.x < n) raw[threadIdx.x] = mine[threadIdx.x];
            __syncthreads();
            if ((int)threadIdx.x < n) {  // rows are distinct: rank = number of smaller rows
                const int v = raw[threadIdx.x];
                int rank = 0;
                for (int j = 0; j < n; ++j) rank += raw[j] < v;
                sorted[rank] = swapped_row(v, swap);
            }
            __syncthreads();
            add_rows(sorted, n);
        }
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            const int col = (c * kBlock + threadIdx.x);
            if (col < h8) {
                OutT* dst = dW + id * h + col * 8;
                if constexpr (sizeof(OutT) == 2) {
                    st_bf16x8(dst, pack8(acc[c]));
                } else {
                    f32x4 lo, hi;
                    if (overwrite) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) { lo[k] = acc[c][k]; hi[k] = acc[c][4 + k]; }
                    } else {
                        lo = *reinterpret_cast<f32x4*>(dst);
                        hi = *reinterpret_cast<f32x4*>(dst + 4);
#pragma unroll
                        for (int k = 0; k < 4; ++k) { lo[k] += acc[c][k]; hi[k] += acc[c][4 + k]; }
                    }
                    *reinterpret_cast<f32x4*>(dst) = lo;
                    *reinterpret_cast<f32x4*>(dst + 4) = hi;
                }
            }
        }
    }
    if (overwrite) {
        // ids that do not occur: zero rows.  Rows are dealt round-robin to the blocks, so that the blocks running at any
        // moment write one contiguous window of the buffer; a block reads the counts of up to kBlock of its rows at once, so
        // that the fill streams instead of waiting for one count per row.
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        for (int64_t v0 = blockIdx.x; v0 < V; v0 += (int64_t)gridDim.x * kBlock) {
            const int64_t left = (V - v0 + gridDim.x - 1) / gridDim.x;  // rows v0, v0 + grid, ... below V
            const int m = left < kBlock ? (int)left : kBlock;
            __syncthreads();
            if ((int)threadIdx.x < m) raw[threadIdx.x] = cnt[v0 + (int64_t)threadIdx.x * gridDim.x];
            __syncthreads();
            for (int r = 0; r < m; ++r) {
                if (raw[r] != 0) continue;
                f32x4* dst = reinterpret_cast<f32x4*>(dW + (v0 + (int64_t)r * gridDim.x) * h);
                for (int i = threadIdx.x; i < h * (int)sizeof(OutT) / 16; i += kBlock) __builtin_nontemporal_store(z, dst + i);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Unpadding by a key-padding mask (FlashAttention.forward, llama/transformer.py:117-141: unpad_input / pad_input)
// ---------------------------------------------------------------------------------------------
// mask [rows, s_len] (non-zero = keep), flattened to n = rows * s_len tokens.  One block walks the tokens 1024 at a time
// with a running count:  idx[p] = flat index of the p-th kept token (entries past the last kept token: -1),
// inv[i] = position of token i among the kept ones, or -1;  cu[r + 1] = kept tokens in rows 0..r (cu[0] = 0).
__global__ __launch_bounds__(1024) void mask_compact_kernel(const unsigned char* __restrict__ mask, int64_t n, int s_len,
                                                            int* __restrict__ idx, int* __restrict__ inv, int* __restrict__ cu) {
    __shared__ int wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    int base = 0;
    if (tid == 0) cu[0] = 0;
    for (int64_t i0 = 0; i0 < n; i0 += 1024) {
        const int64_t i = i0 + tid;
        const int m = (i < n && mask[i]) ? 1 : 0;
        int incl = m;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        __syncthreads();  // wsum of the previous round has been read
        if (lane == 63) wsum[wv] = incl;
        __syncthreads();
        int before = 0, total = 0;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            before += k < wv ? wsum[k] : 0;
            total += wsum[k];
        }
        const int upto = base + before + incl;  // kept tokens among 0..i
        if (i < n) {
            inv[i] = m ? upto - 1 : -1;
            if (m) idx[upto - 1] = (int)i;
            if ((i + 1) % s_len == 0) cu[(i + 1) / s_len] = upto;
        }
        base += total;
    }
    for (int64_t i = base + tid; i < n; i += 1024) idx[i] = -1;
}

// out row r = src row idx[r] (zeros where idx[r] is negative or past the source); a row number maps to memory as
// (r / s_len) * batch_stride + (r % s_len) * seq_stride on either side, so [s, b, ...] activations are read and
// written where they lie.
__global__ __launch_bounds__(kBlock) void rows_gather_kernel(const bf16_t* __restrict__ src, const int* __restrict__ idx,
                                                             bf16_t* __restrict__ out, int64_t n_out, int width, int64_t n_src,
                                                             int src_s_len, int64_t src_ss, int64_t src_sb, int out_s_len,
                                                             int64_t out_ss, int64_t out_sb) {
    const int w8 = width >> 3;
    for (int64_t r = blockIdx.x; r < n_out; r += gridDim.x) {
        const int64_t j = idx[r];
        const bool ok = j >= 0 && j < n_src;
        const bf16_t* s = src + (ok ? (j / src_s_len) * src_sb + (j % src_s_len) * src_ss : 0);
        bf16_t* o = out + (r / out_s_len) * out_sb + (r % out_s_len) * out_ss;
        for (int c = threadIdx.x; c < w8; c += kBlock) {
            bf16x8 v;
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = (bf16_t)0.0f;
            if (ok) v = ld_bf16x8(s + c * 8);
            st_bf16x8(o + c * 8, v);
        }
    }
}

// Several tensors copied by one launch: workgroups y copies tensor y.  What it costs at the sizes of a batch's ids and labels is the launch; a copy call
// each is a blit kernel each, and the replay of a captured step waits for all of them (two-layer stack of h = 256, four tensors: 414.6 -> 409.4 us a step).
constexpr int kCopyMax = 8;
struct CopyList {
    const char* src[kCopyMax];
    char* dst[kCopyMax];
    int64_t bytes[kCopyMax];
};
__global__ __launch_bounds__(kBlock) void copy_list_kernel(const CopyList list) {
    const char* src = list.src[blockIdx.y];
    char* dst = list.dst[blockIdx.y];
    const int64_t n = list.bytes[blockIdx.y], step = (int64_t)gridDim.x * kBlock, first = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int64_t vectors = (((uintptr_t)src | (uintptr_t)dst) & 15) == 0 ? n >> 4 : 0;
    for (int64_t i = first; i < vectors; i += step) reinterpret_cast<u32x4*>(dst)[i] = reinterpret_cast<const u32x4*>(src)[i];
    for (int64_t i = vectors * 16 + first; i < n; i += step) dst[i] = src[i];
}

// y[j, i, :] = x[i, j, :]  for x [d0, d1, inner]   (llama/llama.py:157-168,175-179)
__global__ __launch_bounds__(kBlock) void transpose01_kernel(const bf16_t* __restrict__ x, bf16_t* __restrict__ y, int64_t d0,
                                                             int64_t d1, int inner) {
    const int i8 = inner >> 3;
    const int64_t rows = d0 * d1;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int64_t i = r / d1, j = r % d1;
        const bf16_t* src = x + r * inner;
        bf16_t* dst = y + (j * d0 + i) * inner;
        for (int c = threadIdx.x; c < i8; c += kBlock) st_bf16x8(dst + c * 8, ld_bf16x8(src + c * 8));
    }
}

__global__ __launch_bounds__(kBlock) void add_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ b,
                                                     bf16_t* __restrict__ out, int64_t n8) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += (int64_t)gridDim.x * kBlock) {
        float x[8], y[8];
        unpack8(ld_bf16x8(a + i * 8), x);
        unpack8(ld_bf16x8(b + i * 8), y);
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] += y[k];
        st_bf16x8(out + i * 8, pack8(x));
    }
}

__global__ __launch_bounds__(kBlock) void bf16_to_f32_kernel(const bf16_t* __restrict__ in, float* __restrict__ out, int64_t n8) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += (int64_t)gridDim.x * kBlock) {
        float x[8];
        unpack8(ld_bf16x8(in + i * 8), x);
        f32x4 lo = {x[0], x[1], x[2], x[3]}, hi = {x[4], x[5], x[6], x[7]};
        *reinterpret_cast<f32x4*>(out + i * 8) = lo;
        *reinterpret_cast<f32x4*>(out + i * 8 + 4) = hi;
    }
}

__global__ __launch_bounds__(kBlock) void f32_to_bf16_kernel(const float* __restrict__ in, bf16_t* __restrict__ out, int64_t n8) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += (int64_t)gridDim.x * kBlock) {
        const f32x4 lo = *reinterpret_cast<const f32x4*>(in + i * 8), hi = *reinterpret_cast<const f32x4*>(in + i * 8 + 4);
        float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        st_bf16x8(out + i * 8, pack8(x));
    }
}

// out[r, :] = x[r, :] + bias   (column_parallel_linear.py:43-44)
__global__ __launch_bounds__(kBlock) void bias_add_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ bias,
                                                          bf16_t* __restrict__ out, int64_t rows, int n) {
    const int n8 = n >> 3;
    const int64_t items = rows * n8;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < items; i += (int64_t)gridDim.x * kBlock) {
        const int c = (int)(i % n8);
        float a[8], b[8];
        unpack8(ld_bf16x8(x + i * 8), a);
        unpack8(ld_bf16x8(bias + c * 8), b);
#pragma unroll
        for (int k = 0; k < 8; ++k) a[k] += b[k];
        st_bf16x8(out + i * 8, pack8(a));
    }
}

// partial[blockIdx.y][col] = sum over rows r = blockIdx.y, blockIdx.y + gridDim.y, ... of dy[r][col]   (:100)
__global__ __launch_bounds__(kBlock) void bias_grad_partial_kernel(const bf16_t* __restrict__ dy, float* __restrict__ partial,
                                                                   int64_t rows, int n) {
    const int col = (blockIdx.x * kBlock + threadIdx.x) * 8;
    if (col >= n) return;
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t r = blockIdx.y; r < rows; r += gridDim.y) {
        float v[8];
        unpack8(ld_bf16x8(dy + r * n + col), v);
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] += v[k];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) partial[(int64_t)blockIdx.y * n + col + k] = acc[k];
}

// q / k / v projections (rows of nq, nk, nk heads) + their biases, q and k rotated: bias_add (rounded to bf16) and the rotation
// above in one pass.  An item is 8 low-half + 8 high-half elements of one head of one row.
struct QkvBias {
    const bf16_t *x[3], *bias[3];
    bf16_t* out[3];
};
__global__ __launch_bounds__(kBlock) void bias_rope_kernel(const QkvBias a, const float* __restrict__ cosb, const float* __restrict__ sinb,
                                                           const int64_t* __restrict__ position_ids, int64_t rows, int s, int b, int nq,
                                                           int nk, int d, int64_t npos) {
    const int half = d >> 1, per_head = half >> 3, nheads = nq + 2 * nk;
    const int64_t items = rows * nheads * per_head;
    for (int64_t it = (int64_t)blockIdx.x * kBlock + threadIdx.x; it < items; it += (int64_t)gridDim.x * kBlock) {
        const int j8 = (int)(it % per_head);
        const int64_t rh = it / per_head;
        int head = (int)(rh % nheads);
        const int64_t row = rh / nheads;
        const int which = head < nq ? 0 : (head < nq + nk ? 1 : 2);
        head -= which == 0 ? 0 : (which == 1 ? nq : nq + nk);
        const int col = head * d + j8 * 8;
        const int64_t at = row * (int64_t)((which == 0 ? nq : nk) * d) + col;
        const bf16_t* x = which == 0 ? a.x[0] : (which == 1 ? a.x[1] : a.x[2]);
        const bf16_t* bias = which == 0 ? a.bias[0] : (which == 1 ? a.bias[1] : a.bias[2]);
        bf16_t* out = which == 0 ? a.out[0] : (which == 1 ? a.out[1] : a.out[2]);
        float lo[8], hi[8], bl[8], bh[8];
        unpack8(ld_bf16x8(x + at), lo);
        unpack8(ld_bf16x8(x + at + half), hi);
        unpack8(ld_bf16x8(bias + col), bl);
        unpack8(ld_bf16x8(bias + col + half), bh);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            lo[k] = (float)(bf16_t)(lo[k] + bl[k]);
            hi[k] = (float)(bf16_t)(hi[k] + bh[k]);
        }
        if (which < 2) {
            int64_t pos = position_ids ? position_ids[(row % b) * s + row / b] : row / b;
            pos = pos < 0 ? 0 : (pos >= npos ? npos - 1 : pos);
            const float *cp = cosb + pos * half + j8 * 8, *sp = sinb + pos * half + j8 * 8;
            const f32x4 c0 = *reinterpret_cast<const f32x4*>(cp), c1 = *reinterpret_cast<const f32x4*>(cp + 4);
            const f32x4 s0 = *reinterpret_cast<const f32x4*>(sp), s1 = *reinterpret_cast<const f32x4*>(sp + 4);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float cs = k < 4 ? c0[k] : c1[k - 4], sn = k < 4 ? s0[k] : s1[k - 4];
                const float x1 = lo[k], x2 = hi[k];
                lo[k] = x1 * cs - x2 * sn;
                hi[k] = x2 * cs + x1 * sn;
            }
        }
        st_bf16x8(out + at, pack8(lo));
        st_bf16x8(out + at + half, pack8(hi));
    }
}

// the column sums of a [rows, qw + 2 kw] partial table, written to three targets
// Bound by the latency of its loads: a thread per column walked 64 partial rows one after the other (19.2 us at 1536 columns); now
// 16 threads share a column, four loads each, and meet in LDS (3.0 us).
__global__ __launch_bounds__(kColsumThreads) void qkv_bias_fold_kernel(const float* __restrict__ partial, int nrows, int qw, int kw, const QkvBiasGrad g) {
    constexpr int G = kColsumThreads / 64;
    __shared__ float sums[G][64];
    const int ncols = qw + 2 * kw, lane = threadIdx.x & 63, group = threadIdx.x >> 6, col = blockIdx.x * 64 + lane;
    float acc = 0.f;  // in the order of ezl_colsum_kernel: 16 interleaved groups of rows, then the groups
    if (col < ncols) {
#pragma unroll 4
        for (int r = group; r < nrows; r += G) acc += partial[(size_t)r * ncols + col];
    }
    sums[group][lane] = acc;
    __syncthreads();
    if (group != 0 || col >= ncols) return;
    acc = 0.f;
#pragma unroll
    for (int i = 0; i < G; ++i) acc += sums[i][lane];
    const int which = col < qw ? 0 : (col < qw + kw ? 1 : 2);
    const int c = col - (which == 0 ? 0 : (which == 1 ? qw : qw + kw));
    float* f = which == 0 ? g.f32[0] : (which == 1 ? g.f32[1] : g.f32[2]);
    bf16_t* h = which == 0 ? g.bf16[0] : (which == 1 ? g.bf16[1] : g.bf16[2]);
    const int accumulate = which == 0 ? g.accumulate[0] : (which == 1 ? g.accumulate[1] : g.accumulate[2]);
    if (f) f[c] = accumulate ? f[c] + acc : acc;
    else if (h) h[c] = (bf16_t)acc;
}

}  // namespace

int qkv_bias_rope(const void* const* x, const void* const* bias, void* const* out, int64_t nq, int64_t nk, int64_t d, const void* cos_table,
                  const void* sin_table, const void* position_ids, int64_t s, int64_t b, int64_t npos, hipStream_t stream) {
    EZL_REQUIRE(d % 16 == 0 && npos >= 1 && (position_ids || npos >= s) && cos_table && sin_table, EZL_EUNSUPPORTED,
                "q / k / v bias + rotation: bad head dim or rotary tables");
    QkvBias a;
    for (int i = 0; i < 3; ++i) {
        EZL_REQUIRE(x[i] && bias[i] && out[i] && ezl_aligned16(x[i]) && ezl_aligned16(bias[i]) && ezl_aligned16(out[i]), EZL_EINVAL,
                    "q / k / v bias + rotation: null or misaligned pointer");
        a.x[i] = (const bf16_t*)x[i]; a.bias[i] = (const bf16_t*)bias[i]; a.out[i] = (bf16_t*)out[i];
    }
    hipLaunchKernelGGL(bias_rope_kernel, dim3(grid_for(s * b * (nq + 2 * nk) * (d / 16), kBlock)), dim3(kBlock), 0, stream, a,
                       (const float*)cos_table, (const float*)sin_table, (const int64_t*)position_ids, s * b, (int)s, (int)b, (int)nq,
                       (int)nk, (int)d, npos);
    EZL_LAUNCH_CHECK("q / k / v bias + rotation");
    return EZL_OK;
}

int qkv_bias_grad(const void* dqkv, const QkvBiasGrad& g, int64_t rows, int64_t qw, int64_t kw, void* workspace, hipStream_t stream) {
    const int64_t n = qw + 2 * kw;
    const dim3 grid((unsigned)((n / 8 + kBlock - 1) / kBlock), 64);
    hipLaunchKernelGGL(bias_grad_partial_kernel, grid, dim3(kBlock), 0, stream, (const bf16_t*)dqkv, (float*)workspace, rows, (int)n);
    hipLaunchKernelGGL(qkv_bias_fold_kernel, dim3((unsigned)((n + 63) / 64)), dim3(kColsumThreads), 0, stream, (const float*)workspace, 64, (int)qw,
                       (int)kw, g);
    EZL_LAUNCH_CHECK("q / k / v bias gradient");
    return EZL_OK;
}

extern "C" int ezl_swiglu_fwd(const void* gate, const void* up, void* out, int64_t n, void* stream) {
    EZL_REQUIRE(n >= 0 && n % 8 == 0, EZL_EUNSUPPORTED, "ezl_swiglu_fwd: n must be a multiple of 8");
    EZL_REQUIRE(ezl_aligned16(gate) && ezl_aligned16(up) && ezl_aligned16(out) && (n == 0 || (gate && up && out)), EZL_EINVAL,
                "ezl_swiglu_fwd: null or misaligned pointer");
    if (n == 0) return EZL_OK;
    hipLaunchKernelGGL(ezl_streams(n * 2) ? swiglu_fwd_kernel<true> : swiglu_fwd_kernel<false>, dim3(grid_for(n / 8, kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                       (const bf16_t*)gate, (const bf16_t*)up, (bf16_t*)out, n / 8);
    EZL_LAUNCH_CHECK("ezl_swiglu_fwd");
    return EZL_OK;
}

extern "C" int ezl_swiglu_bwd(const void* dout, const void* gate, const void* up, void* dgate, void* dup, int64_t n,
                              void* stream) {
    EZL_REQUIRE(n >= 0 && n % 8 == 0, EZL_EUNSUPPORTED, "ezl_swiglu_bwd: n must be a multiple of 8");
    EZL_REQUIRE(ezl_aligned16(dout) && ezl_aligned16(gate) && ezl_aligned16(up) && ezl_aligned16(dgate) && ezl_aligned16(dup) &&
                    (n == 0 || (dout && gate && up && dgate && dup)),
                EZL_EINVAL, "ezl_swiglu_bwd: null or misaligned pointer");
    if (n == 0) return EZL_OK;
    hipLaunchKernelGGL(ezl_streams(n * 4) ? swiglu_bwd_kernel<true> : swiglu_bwd_kernel<false>, dim3(grid_for(n / 8, kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                       (const bf16_t*)dout, (const bf16_t*)gate, (const bf16_t*)up, (bf16_t*)dgate, (bf16_t*)dup, n / 8);
    EZL_LAUNCH_CHECK("ezl_swiglu_bwd");
    return EZL_OK;
}

extern "C" int ezl_rope_table(const void* inv_freq, void* cos_out, void* sin_out, int64_t npos, int64_t half_dim,
                              float scale_factor, void* stream) {
    EZL_REQUIRE(npos > 0 && half_dim > 0 && scale_factor > 0.f && inv_freq && cos_out && sin_out, EZL_EINVAL,
                "ezl_rope_table: bad argument");
    hipLaunchKernelGGL(rope_table_kernel, dim3(grid_for(npos * half_dim, kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                       (const float*)inv_freq, (float*)cos_out, (float*)sin_out, npos, (int)half_dim, scale_factor);
    EZL_LAUNCH_CHECK("ezl_rope_table");
    return EZL_OK;
}

namespace {
int rope_launch(const char* name, const void* x0, void* out0, int64_t nh0, int64_t is0, int64_t os0, const void* x1, void* out1,
                int64_t nh1, int64_t is1, int64_t os1, const void* cos_table, const void* sin_table, const void* position_ids,
                int64_t s, int64_t b, int64_t d, int64_t npos, int backward, void* stream) {
    EZL_REQUIRE(s >= 0 && b > 0 && nh0 > 0 && nh1 >= 0 && d > 0 && d % 16 == 0, EZL_EUNSUPPORTED,
                "%s: head dim must be a multiple of 16 (got %lld)", name, (long long)d);
    EZL_REQUIRE(is0 % 8 == 0 && os0 % 8 == 0 && is0 >= nh0 * d && os0 >= nh0 * d, EZL_EINVAL, "%s: bad row stride", name);
    EZL_REQUIRE(nh1 == 0 || (is1 % 8 == 0 && os1 % 8 == 0 && is1 >= nh1 * d && os1 >= nh1 * d), EZL_EINVAL, "%s: bad row stride", name);
    EZL_REQUIRE(npos >= 1 && (position_ids || npos >= s), EZL_EINVAL, "%s: cos/sin table shorter than the sequence", name);
    EZL_REQUIRE((s == 0 || (x0 && out0 && (nh1 == 0 || (x1 && out1)))) && cos_table && sin_table && ezl_aligned16(x0) &&
                    ezl_aligned16(out0) && ezl_aligned16(x1) && ezl_aligned16(out1) && ezl_aligned16(cos_table) &&
                    ezl_aligned16(sin_table),
                EZL_EINVAL, "%s: null or misaligned pointer", name);
    EZL_REQUIRE(s < (1LL << 31) && b < (1LL << 31) && nh0 + nh1 < (1LL << 24), EZL_EUNSUPPORTED, "%s: shape too large", name);
    if (s == 0) return EZL_OK;
    const int64_t items = s * b * (nh0 + nh1) * (d / 16);
    const RopeSide a = {(const bf16_t*)x0, (bf16_t*)out0, is0, os0};
    const RopeSide c = {(const bf16_t*)x1, (bf16_t*)out1, is1, os1};
    hipLaunchKernelGGL(rope_kernel, dim3(grid_for(items, kBlock)), dim3(kBlock), 0, (hipStream_t)stream, a, c,
                       (const float*)cos_table, (const float*)sin_table, (const int64_t*)position_ids, s * b, (int)s, (int)b,
                       (int)nh0, (int)nh1, (int)d, npos, backward ? -1.0f : 1.0f);
    EZL_LAUNCH_CHECK(name);
    return EZL_OK;
}
}  // namespace

extern "C" int ezl_rope_apply(const void* x, void* out, const void* cos_table, const void* sin_table,
                              const void* position_ids, int64_t s, int64_t b, int64_t nheads, int64_t d,
                              int64_t in_row_stride, int64_t out_row_stride, int64_t npos, int backward, void* stream) {
    return rope_launch("ezl_rope_apply", x, out, nheads, in_row_stride, out_row_stride, nullptr, nullptr, 0, 0, 0, cos_table,
                       sin_table, position_ids, s, b, d, npos, backward, stream);
}

extern "C" int ezl_rope_apply_pair(const void* q, void* q_out, int64_t nq, int64_t q_in_stride, int64_t q_out_stride,
                                   const void* k, void* k_out, int64_t nk, int64_t k_in_stride, int64_t k_out_stride,
                                   const void* cos_table, const void* sin_table, const void* position_ids, int64_t s, int64_t b,
                                   int64_t d, int64_t npos, int backward, void* stream) {
    EZL_REQUIRE(nk > 0, EZL_EINVAL, "ezl_rope_apply_pair: the second tensor needs at least one head");
    return rope_launch("ezl_rope_apply_pair", q, q_out, nq, q_in_stride, q_out_stride, k, k_out, nk, k_in_stride, k_out_stride,
                       cos_table, sin_table, position_ids, s, b, d, npos, backward, stream);
}

namespace {

template <bool HOST>
int launch_ids_in_range(const char* name, const void* ids, int64_t n, int64_t limit, void* bad_flag, void* stream) {
    EZL_REQUIRE(n >= 0 && bad_flag && (n == 0 || ids), EZL_EINVAL, "%s: null pointer", name);
    if (n == 0) return EZL_OK;
    hipLaunchKernelGGL((ids_in_range_kernel<HOST>), dim3(grid_for(n, kBlock, 256)), dim3(kBlock), 0, (hipStream_t)stream,
                       (const int64_t*)ids, n, limit, bad_flag);
    EZL_LAUNCH_CHECK(name);
    return EZL_OK;
}

template <bool HOST>
int launch_embed_gather(const char* name, const void* ids, const void* weight, void* out, void* bad_flag, int64_t rows, int64_t h,
                        int64_t vocab, void* stream, const RowSwap& swap = RowSwap{0, 0}) {
    EZL_REQUIRE(rows >= 0 && h > 0 && h % 8 == 0 && h < (1LL << 31) && vocab > 0, EZL_EUNSUPPORTED,
                "%s: h must be a multiple of 8", name);
    EZL_REQUIRE(bad_flag && (rows == 0 || (ids && weight && out)) && ezl_aligned16(weight) && ezl_aligned16(out), EZL_EINVAL,
                "%s: null or misaligned pointer", name);
    if (rows == 0) return EZL_OK;
    hipLaunchKernelGGL((embed_gather_kernel<HOST>), dim3(grid_for((rows + 3) / 4, 1)), dim3(kBlock), 0, (hipStream_t)stream,
                       (const int64_t*)ids, (const bf16_t*)weight, (bf16_t*)out, rows, (int)h, vocab, bad_flag, swap);
    EZL_LAUNCH_CHECK(name);
    return EZL_OK;
}

}  // namespace

extern "C" int ezl_ids_in_range(const void* ids, int64_t n, int64_t limit, void* bad_flag, void* stream) {
    return launch_ids_in_range<false>("ezl_ids_in_range", ids, n, limit, bad_flag, stream);
}

extern "C" int ezl_ids_in_range_host_flag(const void* ids, int64_t n, int64_t limit, void* host_flag, void* stream) {
    return launch_ids_in_range<true>("ezl_ids_in_range_host_flag", ids, n, limit, host_flag, stream);
}

extern "C" int ezl_embed_gather(const void* ids, const void* weight, void* out, void* bad_flag, int64_t rows, int64_t h,
                                int64_t vocab, void* stream) {
    return launch_embed_gather<false>("ezl_embed_gather", ids, weight, out, bad_flag, rows, h, vocab, stream);
}

extern "C" int ezl_embed_gather_host_flag(const void* ids, const void* weight, void* out, void* host_flag, int64_t rows, int64_t h,
                                          int64_t vocab, void* stream) {
    return launch_embed_gather<true>("ezl_embed_gather_host_flag", ids, weight, out, host_flag, rows, h, vocab, stream);
}

namespace {
int embed_swap_check(const char* name, int64_t d0, int64_t d1) {
    EZL_REQUIRE(d0 > 0 && d1 > 0 && d0 < (1LL << 31) && d1 < (1LL << 31) && d0 * d1 < (1LL << 31), EZL_EUNSUPPORTED, "%s: need 0 < d0 * d1 < 2^31",
                name);
    return EZL_OK;
}
}  // namespace

extern "C" int ezl_embed_gather_swapped(const void* ids, const void* weight, void* out, void* bad_flag, int host_flag, int64_t d0, int64_t d1,
                                        int64_t h, int64_t vocab, void* stream) {
    const char* name = "ezl_embed_gather_swapped";
    if (const int rc = embed_swap_check(name, d0, d1)) return rc;
    const RowSwap swap{(int)d0, (int)d1};
    return host_flag ? launch_embed_gather<true>(name, ids, weight, out, bad_flag, d0 * d1, h, vocab, stream, swap)
                     : launch_embed_gather<false>(name, ids, weight, out, bad_flag, d0 * d1, h, vocab, stream, swap);
}

extern "C" int64_t ezl_embed_scatter_add_workspace_bytes(int64_t rows, int64_t vocab) {
    if (rows < 0 || vocab <= 0) return -1;
    return (4 * vocab + rows + 4 + embed_heavy_max(rows)) * (int64_t)sizeof(int);
}

namespace {
template <typename OutT>
int embed_gradient(const char* name, const void* ids, const void* dy, void* dweight, void* workspace, int64_t workspace_bytes, int64_t rows,
                   int64_t h, int64_t vocab, int accumulate, void* stream, const RowSwap& swap = RowSwap{0, 0}) {
    EZL_REQUIRE(rows >= 0 && h > 0 && h % 8 == 0 && h < (1LL << 31) && vocab > 0, EZL_EUNSUPPORTED,
                "%s: h must be a multiple of 8", name);
    EZL_REQUIRE((rows == 0 || (ids && dy && dweight)) && ezl_aligned16(dy), EZL_EINVAL,
                "%s: null or misaligned pointer", name);
    if (rows == 0 && accumulate) return EZL_OK;
    EZL_REQUIRE(dweight, EZL_EINVAL, "%s: null or misaligned pointer", name);
    EZL_REQUIRE(h <= 8192 * 2, EZL_EUNSUPPORTED, "%s: h must be <= 16384", name);
    EZL_REQUIRE(rows < (1LL << 31) && vocab < (1LL << 31), EZL_EUNSUPPORTED, "%s: more than 2^31 rows or ids", name);
    EZL_REQUIRE(((uintptr_t)dweight & 15) == 0, EZL_EINVAL, "%s: dweight must be 16-byte aligned", name);
    EZL_REQUIRE(workspace && ((uintptr_t)workspace & 3) == 0 && workspace_bytes >= ezl_embed_scatter_add_workspace_bytes(rows, vocab),
                EZL_EINVAL, "%s: workspace missing or smaller than ezl_embed_scatter_add_workspace_bytes()", name);
    int* cnt = (int*)workspace;
    int* first = cnt + vocab;
    int* off = first + vocab;
    int* fill = off + vocab;
    int* bucket = fill + vocab;
    int* cursor = bucket + rows;
    int* heavy = cursor + 4;
    hipStream_t st = (hipStream_t)stream;
    // one workgroup per token row (accumulate) or per vocabulary row, whichever is more: the zero fill of the rows that
    // received nothing is most of the traffic when the result overwrites the buffer
    // Overwriting a large table ([152064, 5120] fp32 = 3.1 GB, say) is mostly a zero fill, and a flat fill kernel in front
    // of the adding form writes it faster than the per-row fill inside the scatter kernel does (measured 502 against 580 us
    // at that size); for a table of 0.5 GB the fused form wins (99 against 116 us) because the two parts overlap.
    const bool flat_fill = !accumulate && vocab * h * (int64_t)sizeof(OutT) >= (int64_t)1 << 30;
    if (flat_fill) {
        const int64_t n4 = vocab * h * (int64_t)sizeof(OutT) / 16;
        hipLaunchKernelGGL(zero_f32x4_kernel, dim3(grid_for(n4, 4 * kBlock, (int64_t)1 << 20)), dim3(kBlock), 0, st, (f32x4*)dweight, n4);
    }
    const int overwrite = accumulate || flat_fill ? 0 : 1;
    if (overwrite ? rows <= kSmallRowsZero && vocab <= kSmallVocab : rows <= kSmallRows) {
        hipLaunchKernelGGL(embed_tables_small_kernel, dim3(1), dim3(kSmallThreads), 0, st, (const int64_t*)ids, cnt, first, off, bucket, cursor,
                           heavy, (int)rows, vocab, overwrite);
    } else {
        hipLaunchKernelGGL(embed_tables_init_kernel, dim3(grid_for(vocab, kBlock, 1024)), dim3(kBlock), 0, st, cnt, first, fill, cursor, vocab);
        hipLaunchKernelGGL(embed_count_kernel, dim3(grid_for(rows, kBlock, 1024)), dim3(kBlock), 0, st, (const int64_t*)ids, cnt, first,
                           rows, vocab);
        hipLaunchKernelGGL(embed_assign_kernel, dim3(grid_for(rows, kBlock, 1024)), dim3(kBlock), 0, st, (const int64_t*)ids, cnt, first, off,
                           cursor, heavy, rows, vocab);
        hipLaunchKernelGGL(embed_bucket_kernel, dim3(grid_for(rows, kBlock, 1024)), dim3(kBlock), 0, st, (const int64_t*)ids, off, fill,
                           bucket, rows, vocab);
    }
    EZL_LAUNCH_CHECK(name);
    const dim3 grid(grid_for(overwrite ? (rows > vocab ? rows : vocab) : rows, 1));
    if (h <= 8 * kBlock * 2)
        hipLaunchKernelGGL((embed_scatter_bucket_kernel<2, OutT>), grid, dim3(kBlock), 0, st, (const int64_t*)ids, (const bf16_t*)dy,
                           (OutT*)dweight, cnt, first, off, bucket, cursor, heavy, rows, (int)h, vocab, overwrite, swap);
    else if (h <= 8 * kBlock * 4)
        hipLaunchKernelGGL((embed_scatter_bucket_kernel<4, OutT>), grid, dim3(kBlock), 0, st, (const int64_t*)ids, (const bf16_t*)dy,
                           (OutT*)dweight, cnt, first, off, bucket, cursor, heavy, rows, (int)h, vocab, overwrite, swap);
    else
        hipLaunchKernelGGL((embed_scatter_bucket_kernel<8, OutT>), grid, dim3(kBlock), 0, st, (const int64_t*)ids, (const bf16_t*)dy,
                           (OutT*)dweight, cnt, first, off, bucket, cursor, heavy, rows, (int)h, vocab, overwrite, swap);
    EZL_LAUNCH_CHECK(name);
    return EZL_OK;
}
}  // namespace

extern "C" int ezl_embed_scatter_add(const void* ids, const void* dy, void* dweight_f32, void* workspace, int64_t workspace_bytes,
                                     int64_t rows, int64_t h, int64_t vocab, int accumulate, void* stream) {
    return embed_gradient<float>("ezl_embed_scatter_add", ids, dy, dweight_f32, workspace, workspace_bytes, rows, h, vocab, accumulate, stream);
}

extern "C" int ezl_embed_grad_bf16(const void* ids, const void* dy, void* dweight_bf16, void* workspace, int64_t workspace_bytes,
                                   int64_t rows, int64_t h, int64_t vocab, void* stream) {
    return embed_gradient<bf16_t>("ezl_embed_grad_bf16", ids, dy, dweight_bf16, workspace, workspace_bytes, rows, h, vocab, 0, stream);
}

extern "C" int ezl_embed_grad_swapped(const void* ids, const void* dy, void* dweight, int fp32, void* workspace, int64_t workspace_bytes, int64_t d0,
                                      int64_t d1, int64_t h, int64_t vocab, int accumulate, void* stream) {
    const char* name = "ezl_embed_grad_swapped";
    if (const int rc = embed_swap_check(name, d0, d1)) return rc;
    EZL_REQUIRE(fp32 || !accumulate, EZL_EUNSUPPORTED, "%s: a bf16 gradient is overwritten", name);
    const RowSwap swap{(int)d0, (int)d1};
    return fp32 ? embed_gradient<float>(name, ids, dy, dweight, workspace, workspace_bytes, d0 * d1, h, vocab, accumulate, stream, swap)
                : embed_gradient<bf16_t>(name, ids, dy, dweight, workspace, workspace_bytes, d0 * d1, h, vocab, 0, stream, swap);
}

extern "C" int ezl_transpose01(const void* x, void* y, int64_t d0, int64_t d1, int64_t inner, void* stream) {
    EZL_REQUIRE(d0 >= 0 && d1 >= 0 && inner > 0 && inner % 8 == 0 && inner < (1LL << 31), EZL_EUNSUPPORTED,
                "ezl_transpose01: inner must be a multiple of 8");
    EZL_REQUIRE((d0 * d1 == 0 || (x && y)) && ezl_aligned16(x) && ezl_aligned16(y), EZL_EINVAL,
                "ezl_transpose01: null or misaligned pointer");
    if (d0 * d1 == 0) return EZL_OK;
    hipLaunchKernelGGL(transpose01_kernel, dim3(grid_for(d0 * d1, 1)), dim3(kBlock), 0, (hipStream_t)stream, (const bf16_t*)x,
                       (bf16_t*)y, d0, d1, (int)inner);
    EZL_LAUNCH_CHECK("ezl_transpose01");
    return EZL_OK;
}

extern "C" int ezl_copy_list(int count, const void* const* src, void* const* dst, const int64_t* bytes, void* stream) {
    EZL_REQUIRE(count >= 0 && (count == 0 || (src && dst && bytes)), EZL_EINVAL, "ezl_copy_list: bad count or null argument array");
    for (int i = 0; i < count; ++i)
        EZL_REQUIRE(bytes[i] >= 0 && (bytes[i] == 0 || (src[i] && dst[i])), EZL_EINVAL, "ezl_copy_list: negative size or null pointer");
    for (int at = 0; at < count; at += kCopyMax) {
        CopyList list = {};
        const int n = count - at < kCopyMax ? count - at : kCopyMax;
        int64_t most = 0;
        for (int i = 0; i < n; ++i) {
            list.src[i] = (const char*)src[at + i];
            list.dst[i] = (char*)dst[at + i];
            list.bytes[i] = bytes[at + i];
            most = bytes[at + i] > most ? bytes[at + i] : most;
        }
        if (most == 0) continue;
        hipLaunchKernelGGL(copy_list_kernel, dim3(grid_for((most + 15) / 16, kBlock, 1024), (unsigned)n), dim3(kBlock), 0, (hipStream_t)stream, list);
        EZL_LAUNCH_CHECK("ezl_copy_list");
    }
    return EZL_OK;
}

extern "C" int ezl_add(const void* a, const void* b, void* out, int64_t n, void* stream) {
    EZL_REQUIRE(n >= 0 && n % 8 == 0, EZL_EUNSUPPORTED, "ezl_add: n must be a multiple of 8");
    EZL_REQUIRE((n == 0 || (a && b && out)) && ezl_aligned16(a) && ezl_aligned16(b) && ezl_aligned16(out), EZL_EINVAL,
                "ezl_add: null or misaligned pointer");
    if (n == 0) return EZL_OK;
    hipLaunchKernelGGL(add_kernel, dim3(grid_for(n / 8, kBlock)), dim3(kBlock), 0, (hipStream_t)stream, (const bf16_t*)a,
                       (const bf16_t*)b, (bf16_t*)out, n / 8);
    EZL_LAUNCH_CHECK("ezl_add");
    return EZL_OK;
}

extern "C" int ezl_cast_bf16_to_f32(const void* in, void* out, int64_t n, void* stream) {
    EZL_REQUIRE(n >= 0 && n % 8 == 0, EZL_EUNSUPPORTED, "ezl_cast_bf16_to_f32: n must be a multiple of 8");
    EZL_REQUIRE((n == 0 || (in && out)) && ezl_aligned16(in) && ezl_aligned16(out), EZL_EINVAL,
                "ezl_cast_bf16_to_f32: null or misaligned pointer");
    if (n == 0) return EZL_OK;
    hipLaunchKernelGGL(bf16_to_f32_kernel, dim3(grid_for(n / 8, kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                       (const bf16_t*)in, (float*)out, n / 8);
    EZL_LAUNCH_CHECK("ezl_cast_bf16_to_f32");
    return EZL_OK;
}

extern "C" int ezl_cast_f32_to_bf16(const void* in, void* out, int64_t n, void* stream) {
    EZL_REQUIRE(n >= 0 && n % 8 == 0, EZL_EUNSUPPORTED, "ezl_cast_f32_to_bf16: n must be a multiple of 8");
    EZL_REQUIRE((n == 0 || (in && out)) && ezl_aligned16(in) && ezl_aligned16(out), EZL_EINVAL,
                "ezl_cast_f32_to_bf16: null or misaligned pointer");
    if (n == 0) return EZL_OK;
    hipLaunchKernelGGL(f32_to_bf16_kernel, dim3(grid_for(n / 8, kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                       (const float*)in, (bf16_t*)out, n / 8);
    EZL_LAUNCH_CHECK("ezl_cast_f32_to_bf16");
    return EZL_OK;
}

extern "C" int ezl_bias_add(const void* x, const void* bias, void* out, int64_t rows, int64_t n, void* stream) {
    EZL_REQUIRE(rows >= 0 && n > 0 && n % 8 == 0 && n < (1LL << 31), EZL_EUNSUPPORTED, "ezl_bias_add: n must be a multiple of 8");
    EZL_REQUIRE((rows == 0 || (x && bias && out)) && ezl_aligned16(x) && ezl_aligned16(bias) && ezl_aligned16(out), EZL_EINVAL,
                "ezl_bias_add: null or misaligned pointer");
    if (rows == 0) return EZL_OK;
    hipLaunchKernelGGL(bias_add_kernel, dim3(grid_for(rows * (n / 8), kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                       (const bf16_t*)x, (const bf16_t*)bias, (bf16_t*)out, rows, (int)n);
    EZL_LAUNCH_CHECK("ezl_bias_add");
    return EZL_OK;
}

extern "C" int64_t ezl_bias_grad_workspace_bytes(int64_t rows, int64_t n) {
    (void)rows;
    return (int64_t)64 * n * (int64_t)sizeof(float);
}

extern "C" int ezl_bias_grad(const void* dy, void* db_bf16, void* db_f32, int accumulate, void* workspace,
                             int64_t workspace_bytes, int64_t rows, int64_t n, void* stream) {
    EZL_REQUIRE(rows >= 0 && n > 0 && n % 8 == 0 && n < (1LL << 31), EZL_EUNSUPPORTED, "ezl_bias_grad: n must be a multiple of 8");
    EZL_REQUIRE(dy && workspace && ezl_aligned16(dy) && ((db_bf16 != nullptr) != (db_f32 != nullptr)), EZL_EINVAL,
                "ezl_bias_grad: bad pointer arguments");
    EZL_REQUIRE(workspace_bytes >= ezl_bias_grad_workspace_bytes(rows, n), EZL_EINVAL, "ezl_bias_grad: workspace too small");
    const dim3 grid((unsigned)((n / 8 + kBlock - 1) / kBlock), 64);
    hipLaunchKernelGGL(bias_grad_partial_kernel, grid, dim3(kBlock), 0, (hipStream_t)stream, (const bf16_t*)dy, (float*)workspace,
                       rows, (int)n);
    EZL_LAUNCH_CHECK("ezl_bias_grad");
    hipLaunchKernelGGL(ezl_colsum_kernel<0>, dim3((unsigned)((n + 63) / 64)), dim3(kColsumThreads), 0, (hipStream_t)stream,
                       (const float*)workspace, 64, (int)n, (bf16_t*)db_bf16, (float*)db_f32, accumulate);
    EZL_LAUNCH_CHECK("ezl_bias_grad(colsum)");
    return EZL_OK;
}

extern "C" int ezl_mask_compact(const void* mask_u8, int64_t rows, int64_t s_len, void* idx, void* inv, void* cu_seqlens, void* stream) {
    EZL_REQUIRE(rows >= 0 && s_len > 0 && rows * s_len < (1LL << 31), EZL_EINVAL, "ezl_mask_compact: bad shape");
    EZL_REQUIRE(cu_seqlens && (rows == 0 || (mask_u8 && idx && inv)), EZL_EINVAL, "ezl_mask_compact: null pointer");
    hipLaunchKernelGGL(mask_compact_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, (const unsigned char*)mask_u8, rows * s_len,
                       (int)s_len, (int*)idx, (int*)inv, (int*)cu_seqlens);
    EZL_LAUNCH_CHECK("ezl_mask_compact");
    return EZL_OK;
}

extern "C" int ezl_rows_gather(const void* src, const void* idx, void* out, int64_t n_out, int64_t width, int64_t n_src,
                               int64_t src_s_len, int64_t src_seq_stride, int64_t src_batch_stride, int64_t out_s_len,
                               int64_t out_seq_stride, int64_t out_batch_stride, void* stream) {
    EZL_REQUIRE(n_out >= 0 && n_src >= 0 && width > 0 && width % 8 == 0 && width < (1LL << 31), EZL_EUNSUPPORTED,
                "ezl_rows_gather: width must be a multiple of 8");
    EZL_REQUIRE(src_s_len > 0 && out_s_len > 0 && src_s_len < (1LL << 31) && out_s_len < (1LL << 31) && src_seq_stride % 8 == 0 &&
                    src_batch_stride % 8 == 0 && out_seq_stride % 8 == 0 && out_batch_stride % 8 == 0,
                EZL_EINVAL, "ezl_rows_gather: strides must be multiples of 8 elements");
    EZL_REQUIRE((n_out == 0 || (idx && out && (src || n_src == 0))) && ezl_aligned16(src) && ezl_aligned16(out), EZL_EINVAL,
                "ezl_rows_gather: null or misaligned pointer");
    if (n_out == 0) return EZL_OK;
    hipLaunchKernelGGL(rows_gather_kernel, dim3(grid_for(n_out, 1)), dim3(kBlock), 0, (hipStream_t)stream, (const bf16_t*)src,
                       (const int*)idx, (bf16_t*)out, n_out, (int)width, n_src, (int)src_s_len, src_seq_stride, src_batch_stride,
                       (int)out_s_len, out_seq_stride, out_batch_stride);
    EZL_LAUNCH_CHECK("ezl_rows_gather");
    return EZL_OK;
}
