// Attention for launches that leave the chip idle with attention.hip's blocks of 128 queries or keys.
//
// A workgroup there walks all tiles that its 128 rows see, one after the other, and a tile takes a wave 1.2 - 1.6 us however few
// workgroups there are: 2 x 512 tokens with 4 heads are 32 workgroups on 256 CUs, the longest of 8 tiles: 13 - 15 us per kernel.
// Here a workgroup owns 32 rows, and its waves share out the tiles that these see: wave w takes tiles w, w + NW, ..., each out
// of its own piece of LDS with no barrier in the loop, and the waves' sums are added in wave order at the end (forward: after
// they are brought to a common reference point).  That is four times the workgroups and a chain a quarter (an eighth) as long, for four times
// the reads of K / V (Q / dO), which come from L2.  dQ and dK/dV, which need nothing of each other once both compute
// delta = rowsum(dO * O) for themselves, go out in one launch.
// One LDS array per kernel, fragment reads through restrict-qualified pointers (see attention_tile.h on what the compiler does
// otherwise): the waits for a wave's own tile loads are explicit.
#include "attention_tile.h"

namespace {

// rows of a tile from global memory into a wave's own LDS piece, ROWS at a time (rows past `last` re-read it)
template <int D, int ROWS>
struct WaveTile {
    static constexpr int LD = Tile<D>::LD;
    static constexpr int NQ = (ROWS * LD * 2 + 1023) / 1024;  // 1 KiB wave loads
    static constexpr int ELEMS = NQ * 512;
    static __device__ __forceinline__ void load(const bf16_t* rows, int64_t ss, int last, bf16_t* stage, int lane) {
        const __amdgpu_buffer_rsrc_t g =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(rows)), 0, 0xffffffffu, 0x00020000);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int byte = q * 1024 + lane * 16;
            int row = byte / (LD * 2);
            int colb = byte - row * (LD * 2);
            colb = colb < D * 2 ? colb : 0;
            row = row < last ? row : last;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(g, (lds_void*)(stage + q * 512), 16, (uint32_t)row * (uint32_t)(ss * 2) + (uint32_t)colb, 0, 0, 0);
        }
    }
};

__device__ __forceinline__ void wait_tile() {  // this wave's loads have landed
    __builtin_amdgcn_s_waitcnt(0x0F70);        // vmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void wait_reads() {  // this wave's LDS reads are done: its tile may be overwritten
    __builtin_amdgcn_s_waitcnt(0xC07F);         // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
}
// a wave's tile memory, made opaque: the fragment reads are restrict-qualified, so a refilled tile must not look like the same address
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+s"(x));
    return x;
}
template <int N>
__device__ __forceinline__ void zero(f32x16 (&a)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) a[i][r] = 0.f;
}
// registers 4 i .. 4 i + 3 of an array of accumulator blocks
template <int N>
__device__ __forceinline__ f32x4 quad(const f32x16 (&a)[N], int i) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = a[i >> 2][(i & 3) * 4 + e];
    return v;
}

// =================================================================================================
// forward: 32 queries of one head
// =================================================================================================
// K fragments go straight from global memory into registers (their reduction index is contiguous), V through LDS for the
// transposing reads.
template <int D, int NW>
__global__ __launch_bounds__(NW * 64) void attn_fwd_small_kernel(AttnParams p) {
    using TL = Tile<D>;
    using WT = WaveTile<D, 64>;
    constexpr int KD = D / 16, NB = D / 32;
    static_assert(WT::ELEMS * 2 >= NB * 16 * 64 * 4 + 2 * 64 * 4, "a wave's sums and statistics fit its tile memory");
    __shared__ __attribute__((aligned(1024))) bf16_t smem[NW * WT::ELEMS + 2 * kFindBlockInts];
    int doc_start, doc_len, qb, rank, hq;
    heads_of(blockIdx.x, p.nq, rank, hq);
    if (!find_block(p.cu, p.ndocs, p.s_len, p.T, rank, 32, doc_start, doc_len, qb, reinterpret_cast<int*>(smem + NW * WT::ELEMS))) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hk = hq / (p.nq / p.nk);
    const int q0 = qb * 32, qi = q0 + (lane & 31);
    const int kend = q0 + 32 < doc_len ? q0 + 32 : doc_len;
    const int ntiles = (kend + 63) / 64;
    const bf16_t* kbase = p.k + tok_off(doc_start, p.s_len, p.k_ss, p.k_sb) + (int64_t)hk * D;
    const bf16_t* vbase = p.v + tok_off(doc_start, p.s_len, p.v_ss, p.v_sb) + (int64_t)hk * D;
    bf16_t* tile = smem + wave * WT::ELEMS;

    bf16x8 qf[KD], kf[2][KD];
    auto load_k = [&](int t) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            int row = t * 64 + kb * 32 + (lane & 31);
            row = row < doc_len ? row : doc_len - 1;
            load_row_frags<D>(kbase + (int64_t)row * p.k_ss, lane, kf[kb]);
        }
    };
    auto load_v = [&](int t) { WT::load(vbase + (int64_t)t * 64 * p.v_ss, p.v_ss, doc_len - 1 - t * 64, tile, lane); };
    if (wave < ntiles) {
        load_k(wave);
        load_v(wave);
    }
    load_row_frags<D>(p.q + tok_off(doc_start + (qi < doc_len ? qi : doc_len - 1), p.s_len, p.q_ss, p.q_sb) + (int64_t)hq * D, lane, qf);

    f32x16 oacc[NB];
    zero(oacc);
    float m = -INFINITY, lsum = 0.f;
    const float sl2 = p.scale * kLog2e;
    for (int t = wave; t < ntiles; t += NW) {
        const int key0 = t * 64;
        f32x16 s[2];
        zero(s);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < KD; ++i) s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kb][i], qf[i], s[kb], 0, 0, 0);
        if (t + NW < ntiles) load_k(t + NW);
        if (key0 + 63 > q0) {  // the tile meets the diagonal
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (key0 + kb * 32 + acc_row(r, lane) > qi) s[kb][r] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mnew = fmaxf(m, mx), ref = mnew == -INFINITY ? 0.f : mnew;
        const float alpha = __builtin_amdgcn_exp2f((m - ref) * sl2);  // m = -inf: 0
        m = mnew;
        lsum *= alpha;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[i][r] *= alpha;
        const float moff = ref * sl2;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[kb][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r], sl2, -moff));
                lsum += s[kb][r];
            }
        wait_tile();
        const bf16_t* sV = smem + opaque(wave * WT::ELEMS);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const bf16x8 pf = acc_to_b(s[g >> 1], g & 1);
#pragma unroll
            for (int db = 0; db < NB; ++db)
                oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::frag_tr(sV, g * 16, db * 32, lane), pf, oacc[db], 0, 0, 0);
        }
        wait_reads();
        if (t + NW < ntiles) load_v(t + NW);
    }
    lsum += __shfl_xor(lsum, 32, 64);
    // the waves' sums, brought to the common reference point and added in wave order; a wave finishes every NW-th quad of registers
    float* sums = reinterpret_cast<float*>(smem);
    constexpr int PIECE = WT::ELEMS / 2, STAT = NB * 16 * 64;  // floats per wave; its statistics behind its sums
#pragma unroll
    for (int i = 0; i < NB * 4; ++i) *reinterpret_cast<f32x4*>(sums + wave * PIECE + (i * 64 + lane) * 4) = quad(oacc, i);
    sums[wave * PIECE + STAT + lane] = m;
    sums[wave * PIECE + STAT + 64 + lane] = lsum;
    __syncthreads();
    float mw[NW], mtot = -INFINITY, ltot = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        mw[w] = sums[w * PIECE + STAT + lane];
        mtot = fmaxf(mtot, mw[w]);
    }
    const float ref = mtot == -INFINITY ? 0.f : mtot;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        mw[w] = __builtin_amdgcn_exp2f((mw[w] - ref) * sl2);
        ltot += mw[w] * sums[w * PIECE + STAT + 64 + lane];
    }
    if (qi >= doc_len) return;
    const float inv = 1.0f / ltot;
    bf16_t* orow = p.out + tok_off(doc_start + qi, p.s_len, p.o_ss, p.o_sb) + (int64_t)hq * D;
#pragma unroll
    for (int n = 0; n < (NB * 4 + NW - 1) / NW; ++n) {
        const int i = n * NW + wave;
        if (i >= NB * 4) break;
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) o += mw[w] * *reinterpret_cast<const f32x4*>(sums + w * PIECE + (i * 64 + lane) * 4);
        bf16x4 b;
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = (bf16_t)(o[e] * inv);
        *reinterpret_cast<bf16x4*>(orow + (i >> 2) * 32 + 8 * (i & 3) + 4 * (lane >> 5)) = b;
    }
    if (wave == 0 && lane < 32) p.lse[(int64_t)hq * p.T + doc_start + qi] = mtot * p.scale + __builtin_amdgcn_logf(ltot) * kLn2;
}

// =================================================================================================
// backward: workgroups of 32 keys (dK, dV) and of 32 queries (dQ)
// =================================================================================================
// Adds the waves' sums (NB blocks each) in wave order; a wave returns every NW-th quad of registers through out(quad index, sum).
template <int NB, int NW, int PIECE, class Out>
__device__ __forceinline__ void add_waves(float* sums, const f32x16 (&acc)[NB], int wave, int lane, Out&& out) {
#pragma unroll
    for (int i = 0; i < NB * 4; ++i) *reinterpret_cast<f32x4*>(sums + wave * PIECE + (i * 64 + lane) * 4) = quad(acc, i);
    __syncthreads();
#pragma unroll
    for (int n = 0; n < (NB * 4 + NW - 1) / NW; ++n) {
        const int i = n * NW + wave;
        if (i >= NB * 4) break;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) v += *reinterpret_cast<const f32x4*>(sums + w * PIECE + (i * 64 + lane) * 4);
        out(i, v);
    }
}

template <int D, int NW>
struct BwdSmall {
    using TL = Tile<D>;
    using QT = WaveTile<D, 32>;  // dK/dV: Q and dO tiles of 32 queries
    using KT = WaveTile<D, 64>;  // dQ: K tiles of 64 keys
    static constexpr int KD = D / 16, NB = D / 32;
    static constexpr int STAT = 2 * 32 * 2;  // lse | delta of a tile's 32 queries, in bf16 elements
    static constexpr int WAVE = (2 * QT::ELEMS + STAT > KT::ELEMS ? 2 * QT::ELEMS + STAT : KT::ELEMS) / 8 * 8;
    static constexpr int ELEMS = NW * WAVE + 2 * kFindBlockInts;
    static_assert(WAVE * 2 >= NB * 16 * 64 * 4, "a wave's sums of one result fit its tile memory");

    static __device__ __forceinline__ void keys(const AttnParams& p, int lin, bf16_t* smem) {
        int doc_start, doc_len, kbk, rank, hk;
        heads_of(lin, p.nk, rank, hk);
        if (!find_block(p.cu, p.ndocs, p.s_len, p.T, rank, 32, doc_start, doc_len, kbk, reinterpret_cast<int*>(smem + NW * WAVE))) return;
        kbk = (doc_len + 31) / 32 - 1 - kbk;  // rank 0 = most queries to walk = the piece's first keys
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int group = p.nq / p.nk, k0 = kbk * 32, kj = k0 + (lane & 31);
        const int nqt = (doc_len + 31) / 32 - kbk, total = nqt * group;  // (query head of the group, query tile) pairs
        const float sl2 = p.scale * kLog2e;
        const bf16_t* qdoc = p.q + tok_off(doc_start, p.s_len, p.q_ss, p.q_sb);
        const bf16_t* dodoc = p.dout + tok_off(doc_start, p.s_len, p.do_ss, p.do_sb);
        const bf16_t* odoc = p.o + tok_off(doc_start, p.s_len, p.o_ss, p.o_sb);
        bf16_t* tile = smem + wave * WAVE;
        float* stat = reinterpret_cast<float*>(tile + 2 * QT::ELEMS);  // [lse * log2e | delta][query]

        bf16x8 of[KD];  // O of this lane's query (row lane & 31 of the tile), every other 8 columns
        float lse = 0.f;
        auto load = [&](int it) {
            const int hq = hk * group + it / nqt, row0 = (kbk + it % nqt) * 32, last = doc_len - 1 - row0;
            QT::load(qdoc + (int64_t)hq * D + (int64_t)row0 * p.q_ss, p.q_ss, last, tile, lane);
            QT::load(dodoc + (int64_t)hq * D + (int64_t)row0 * p.do_ss, p.do_ss, last, tile + QT::ELEMS, lane);
            int row = lane & 31;
            row = row < last ? row : last;
            load_row_frags<D>(odoc + (int64_t)hq * D + (int64_t)(row0 + row) * p.o_ss, lane, of);
            lse = p.lse[(int64_t)hq * p.T + doc_start + row0 + row];
        };
        if (wave < total) load(wave);
        bf16x8 kf[KD], vf[KD];
        const int krow = kj < doc_len ? kj : doc_len - 1;
        load_row_frags<D>(p.k + tok_off(doc_start + krow, p.s_len, p.k_ss, p.k_sb) + (int64_t)hk * D, lane, kf);
        load_row_frags<D>(p.v + tok_off(doc_start + krow, p.s_len, p.v_ss, p.v_sb) + (int64_t)hk * D, lane, vf);
        f32x16 dk[NB], dv[NB];
        zero(dk);
        zero(dv);
        for (int it = wave; it < total; it += NW) {
            const int qs0 = (kbk + it % nqt) * 32;
            wait_tile();
            const bf16_t* sQ = smem + opaque(wave * WAVE);
            const bf16_t* sdO = sQ + QT::ELEMS;
            f32x16 s[1], dp[1];
            zero(s);
            zero(dp);
            float delta = 0.f;
#pragma unroll
            for (int i = 0; i < KD; ++i) {
                const bf16x8 fq = TL::frag_kc(sQ, 0, i, lane), fo = TL::frag_kc(sdO, 0, i, lane);
                s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fq, kf[i], s[0], 0, 0, 0);
                dp[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fo, vf[i], dp[0], 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 8; ++e) delta += (float)of[i][e] * (float)fo[e];
            }
            delta += __shfl_xor(delta, 32, 64);
            stat[lane] = lane < 32 ? lse * kLog2e : delta;
            __builtin_amdgcn_wave_barrier();
            // accumulator register r <-> query qs0 + acc_row(r); lane <-> key kj
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const int ql = 8 * r4 + 4 * (lane >> 5);
                const f32x4 l4 = *reinterpret_cast<const f32x4*>(stat + ql), d4 = *reinterpret_cast<const f32x4*>(stat + 32 + ql);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = r4 * 4 + e, q = qs0 + ql + e;
                    const float pe = kj > q || q >= doc_len ? 0.f : __builtin_amdgcn_exp2f(__builtin_fmaf(s[0][r], sl2, -l4[e]));
                    s[0][r] = pe;
                    dp[0][r] = pe * (dp[0][r] - d4[e]);
                }
            }
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const bf16x8 pf = acc_to_b(s[0], g), dsf = acc_to_b(dp[0], g);
#pragma unroll
                for (int db = 0; db < NB; ++db) {
                    dv[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::frag_tr(sdO, 16 * g, db * 32, lane), pf, dv[db], 0, 0, 0);
                    dk[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::frag_tr(sQ, 16 * g, db * 32, lane), dsf, dk[db], 0, 0, 0);
                }
            }
            wait_reads();
            if (it + NW < total) load(it + NW);
        }
        float* sums = reinterpret_cast<float*>(smem);
        const bool valid = kj < doc_len;
        bf16_t* dvrow = p.dv + tok_off(doc_start + krow, p.s_len, p.dv_ss, p.dv_sb) + (int64_t)hk * D;
        bf16_t* dkrow = p.dk + tok_off(doc_start + krow, p.s_len, p.dk_ss, p.dk_sb) + (int64_t)hk * D;
        auto store = [&](bf16_t* rowp, int i, f32x4 v, float scale) {
            bf16x4 b;
#pragma unroll
            for (int e = 0; e < 4; ++e) b[e] = (bf16_t)(v[e] * scale);
            if (valid) *reinterpret_cast<bf16x4*>(rowp + (i >> 2) * 32 + 8 * (i & 3) + 4 * (lane >> 5)) = b;
        };
        __syncthreads();
        add_waves<NB, NW, WAVE / 2>(sums, dv, wave, lane, [&](int i, f32x4 v) { store(dvrow, i, v, 1.0f); });
        __syncthreads();
        add_waves<NB, NW, WAVE / 2>(sums, dk, wave, lane, [&](int i, f32x4 v) { store(dkrow, i, v, p.scale); });
    }

    static __device__ __forceinline__ void queries(const AttnParams& p, int lin, bf16_t* smem) {
        int doc_start, doc_len, qb, rank, hq;
        heads_of(lin, p.nq, rank, hq);
        if (!find_block(p.cu, p.ndocs, p.s_len, p.T, rank, 32, doc_start, doc_len, qb, reinterpret_cast<int*>(smem + NW * WAVE))) return;
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int hk = hq / (p.nq / p.nk);
        const int q0 = qb * 32, qi = q0 + (lane & 31), qrow = qi < doc_len ? qi : doc_len - 1;
        const int kend = q0 + 32 < doc_len ? q0 + 32 : doc_len;
        const int ntiles = (kend + 63) / 64;
        const bf16_t* kbase = p.k + tok_off(doc_start, p.s_len, p.k_ss, p.k_sb) + (int64_t)hk * D;
        const bf16_t* vbase = p.v + tok_off(doc_start, p.s_len, p.v_ss, p.v_sb) + (int64_t)hk * D;
        bf16_t* tile = smem + wave * WAVE;
        const float sl2 = p.scale * kLog2e;

        bf16x8 vf[2][KD];
        auto load = [&](int t) {
            KT::load(kbase + (int64_t)t * 64 * p.k_ss, p.k_ss, doc_len - 1 - t * 64, tile, lane);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                int row = t * 64 + kb * 32 + (lane & 31);
                row = row < doc_len ? row : doc_len - 1;
                load_row_frags<D>(vbase + (int64_t)row * p.v_ss, lane, vf[kb]);
            }
        };
        if (wave < ntiles) load(wave);
        bf16x8 qf[KD], dof[KD];
        load_row_frags<D>(p.q + tok_off(doc_start + qrow, p.s_len, p.q_ss, p.q_sb) + (int64_t)hq * D, lane, qf);
        load_row_frags<D>(p.dout + tok_off(doc_start + qrow, p.s_len, p.do_ss, p.do_sb) + (int64_t)hq * D, lane, dof);
        float delta = 0.f;
        {
            bf16x8 of[KD];
            load_row_frags<D>(p.o + tok_off(doc_start + qrow, p.s_len, p.o_ss, p.o_sb) + (int64_t)hq * D, lane, of);
#pragma unroll
            for (int i = 0; i < KD; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) delta += (float)of[i][e] * (float)dof[i][e];
        }
        delta += __shfl_xor(delta, 32, 64);
        const int64_t stat = (int64_t)hq * p.T + doc_start + qrow;
        const float lse2 = p.lse[stat] * kLog2e;
        if (wave == 0 && lane < 32 && qi < doc_len) p.delta[stat] = delta;
        f32x16 dq[NB];
        zero(dq);
        for (int t = wave; t < ntiles; t += NW) {
            const int key0 = t * 64;
            wait_tile();
            const bf16_t* sK = smem + opaque(wave * WAVE);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                f32x16 s[1], dp[1];
                zero(s);
                zero(dp);
#pragma unroll
                for (int i = 0; i < KD; ++i) {
                    s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::frag_kc(sK, kb * 32, i, lane), qf[i], s[0], 0, 0, 0);
                    dp[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[kb][i], dof[i], dp[0], 0, 0, 0);
                }
                // accumulator register r <-> key key0 + 32 kb + acc_row(r); lane <-> query qi
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float pe = key0 + kb * 32 + acc_row(r, lane) > qi ? 0.f : __builtin_amdgcn_exp2f(__builtin_fmaf(s[0][r], sl2, -lse2));
                    dp[0][r] = pe * (dp[0][r] - delta);
                }
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const bf16x8 dsf = acc_to_b(dp[0], g);
#pragma unroll
                    for (int db = 0; db < NB; ++db)
                        dq[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::frag_tr(sK, kb * 32 + 16 * g, db * 32, lane), dsf, dq[db], 0, 0, 0);
                }
            }
            wait_reads();
            if (t + NW < ntiles) load(t + NW);
        }
        __syncthreads();
        bf16_t* dqrow = p.dq + tok_off(doc_start + qrow, p.s_len, p.dq_ss, p.dq_sb) + (int64_t)hq * D;
        add_waves<NB, NW, WAVE / 2>(reinterpret_cast<float*>(smem), dq, wave, lane, [&](int i, f32x4 v) {
            bf16x4 b;
#pragma unroll
            for (int e = 0; e < 4; ++e) b[e] = (bf16_t)(v[e] * p.scale);
            if (qi < doc_len) *reinterpret_cast<bf16x4*>(dqrow + (i >> 2) * 32 + 8 * (i & 3) + 4 * (lane >> 5)) = b;
        });
    }
};

// workgroups 0 .. key_blocks - 1: keys (the longer chains with grouped queries), the others: queries
template <int D, int NW>
__global__ __launch_bounds__(NW * 64) void attn_bwd_small_kernel(AttnParams p, int key_blocks) {
    using B = BwdSmall<D, NW>;
    __shared__ __attribute__((aligned(1024))) bf16_t smem[B::ELEMS];
    const int lin = blockIdx.x;
    if (lin < key_blocks) B::keys(p, lin, smem);
    else B::queries(p, lin - key_blocks, smem);
}

}  // namespace

// Where these kernels win, on whole rows by the number of 128-row blocks of the launch (each four workgroups here) and the rows' length:
// while all workgroups run at once (two per CU at d = 64, one at d = 128, by their registers) a launch takes its longest chain of
// tiles; beyond that it takes the sum, and the larger blocks do the same work with a quarter of the reads.  us, 128-row kernels
// (as attention.hip would launch them) against these, d / heads / documents x length (blocks):
//   forward   d 64:   4 / 2 x 512 (32) 9.9, 7.2; 6 / 4 x 454 (90) 9.8, 8.5; 5 / 2902 (115) 33.6, 29.6; 13 / 3 x 511 (156) 10.9, 13.4; 12 / 2 x 1024
//             (192) 15.6, 19.8
//             d 128:  9 / 236 (18) 10.1, 7.6; 12 / 645 (72) 17.4, 13.3; 4 / 3 x 1281 (124) 24.9, 27.7; 8 / 4 x 512 (128) 14.6, 16.8
//   backward  d 64:   4 / 2 x 512 (32) 16.8, 12.5; 6 / 4 x 454 (90) 17.7, 17.6; 5 / 2902 (115) 71, 57; 18 / 4 x 162 (108) 14.5, 16.2; 13 / 3 x 400
//             (130) 19.5, 21.9
//             d 128:  6 / 2 x 145 (18) 15.8, 11.5; 19 / 2 x 128 (38) 14.2, 16.5; 3 / 4 x 428 (42) 26.8, 20.9; 2 / 3 x 1455 (70) 71, 51; 5 / 8 x 209
//             (70) 19.3, 25.5; 4 / 3 x 1281 (124) 66, 73
// Long rows pay up to 128 blocks (512 workgroups of keys, 512 of queries), not beyond.  Backward, heads / rows x length (128-row blocks), us with two launches, one,
// these:
//   d 64:  1 / 16384 (128) 570, 353, 257; 3 / 8192 (192) 293, 181, 198; 1 / 4 x 8192 (256) 294, 181, 237; 4 / 16384 (512) 621, 609, 868
//   d 128: 1 / 16384 (128) 856, 705, 540; 3 / 8192 (192) 440, 371, 443; 1 / 4 x 8192 (256) 435, 368, 529; 4 / 16384 (512) 1007, 1118, 1987
// A row of up to 64 tokens is one tile, which there is nothing to share out of; one of two tiles gains only while a CU has one workgroup.  Forward, heads /
// rows x length (32-row workgroups):
//   d 64:  4 / 64 (8) 4.9, 5.3; 41 / 3 x 33 (246) 5.0, 5.6; 16 / 4 x 65 (192) 6.2, 5.5; 24 / 4 x 65 (288) 6.3, 6.8; 16 / 4 x 97 (256) 6.6, 5.7; 64 / 2 x 97 (512) 6.6,
//          6.9; 24 / 4 x 128 (384) 7.1, 7.0
//   d 128: 16 / 2 x 33 (64) 5.8, 6.5; 64 / 2 x 64 (256) 6.5, 7.2; 16 / 65 (48) 7.7, 6.8
// A block of keys walks the queries of every head of its group, which the 128-row kernel deals to several workgroups: with more than two heads
// a group only short chains pay.  Query / kv heads, documents x length, us with dQ and dK/dV of 128 rows in one launch against these:
//   d 64:  8 / 1, 2 x 500 23.2, 54.7; 28 / 7, 3 x 83 13.5, 11.2; 14 / 7, 728 27.9, 28.4; 2 / 1, 3 x 561 21.8, 19.4
//   d 128: 4 / 1, 2 x 802 47.5, 67.5 (two launches 62.2); 12 / 3, 175 20.2, 21.6; 32 / 4, 79 17.1, 21.2; 68 / 17, 114 21.6, 18.4; 2 / 1, 4326 189, 165
// Every workgroup of a packed batch first searches the documents for its block, so that four times the workgroups cost more than with whole rows; these
// kernels have to fit the launched ones at once and gain from documents that are long on average.  Heads, documents x length (mean, longest) of one
// row, us with 128-row kernels (two launches backward), key groups / one launch, these:
//   forward   d 64:  8 / 31 (59, 72) 10.5, 11.2, 20.2; 4 / 64 x 64 10.5, 11.8, 13.4; 4 / 8 x 512 17.0, 16.0, 16.8; 1 / 29 (414, 507) 18.1, 17.1, 17.2; 4 / 7 (586, 2132)
//             37.1, 31.2, 27.9
//             d 128: 2 / 32 x 128 14.2, 15.1, 14.5; 2 / 16 x 256 16.3, 16.8, 15.6; 2 / 7 (586, 2132) 45.8, 39.7, 36.3
//   backward  d 64:  4 / 32 x 512 63, 74, 144; 4 / 16 x 256 30.8, 17.9, 31.5; 4 / 7 (586, 2132) 95, 58, 56; 1 / 45 (188, 752) 48, 28.2, 28.3;
//             2 / 8 x 1024 58, 35, 44; 2 / 4 x 4096 165, 111, 163; 2 / 2 x 2048 91, 56, 44
//             d 128: 4 / 64 x 128 42, 47, 127; 2 / 16 x 256 39, 24.5, 34.6; 1 / 16 (320, 736) 63, 43, 33; 2 / 7 (586, 2132) 135, 101, 65;
//             2 / 8 x 1024 80, 59, 93; 2 / 4 x 4096 239, 184, 359; 2 / 2 x 2048 129, 96, 69
bool attn_small_pays(const AttnSizes& z, bool backward) {
    const int64_t length = z.documents ? z.mean_length() : z.s_len, group = z.nq / z.nk;
    auto blocks = [&](int64_t n) { return (z.documents ? z.launched(n) : z.rows() * ((z.s_len + n - 1) / n)) * z.nq; };
    if (!backward) return length > (z.documents ? 255 : 64) && blocks(32) <= (z.d == 64 && length >= 128 ? 512 : 256);
    if (group > 2 && (length + 31) / 32 * group > 16) return false;
    const int64_t limit = (z.documents || z.d == 64 ? 64 : 32) + length / 32;
    return blocks(128) <= (limit < 128 ? limit : 128);
}

void attn_small_fwd(const AttnParams& p, int d, hipStream_t stream) {
    const dim3 grid((unsigned)(((p.T + 31) / 32 + p.ndocs + p.T / p.s_len) * p.nq));
    if (d == 128) hipLaunchKernelGGL((attn_fwd_small_kernel<128, 4>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((attn_fwd_small_kernel<64, 4>), grid, dim3(256), 0, stream, p);
}

void attn_small_bwd(const AttnParams& p, int d, hipStream_t stream) {
    const int blocks = (p.T + 31) / 32 + p.ndocs + p.T / p.s_len;
    const dim3 grid((unsigned)(blocks * (p.nk + p.nq)));
    if (d == 128) hipLaunchKernelGGL((attn_bwd_small_kernel<128, 4>), grid, dim3(256), 0, stream, p, blocks * p.nk);
    else hipLaunchKernelGGL((attn_bwd_small_kernel<64, 4>), grid, dim3(256), 0, stream, p, blocks * p.nk);
}
