// bf16 MFMA GEMM for gfx950: C[M,N] = A * B with fp32 accumulation.
//
// Replaces the three matmuls of the reference's linear layers
// (base_modules/layers/column_parallel_linear.py:42 forward, :68 input gradient, :99 weight
// gradient; row_parallel_linear.py:113; llama/lm_head.py:62):
//   forward   Y[T,out]  = X[T,in]   * W[out,in]^T    A k-contiguous, B k-contiguous
//   dgrad     dX[T,in]  = dY[T,out] * W[out,in]      A k-contiguous, B n-contiguous
//   wgrad     dW[out,in]= dY[T,out]^T * X[T,in]      A m-contiguous, B n-contiguous   (fp32 or bf16 out)
//
// Tiling: 256x256 block tile, K step 64, 8 waves (2x4), each wave owns 128x64.  Operand tiles are double buffered in LDS
// (2 stages x 2 operands x 32 KiB).  An operand whose reduction dimension is the strided one is kept as it lies in
// memory ([k][256]) and read with ds_read_b64_tr_b16 (the LDS transpose read), so nothing is ever transposed in HBM.
//
// Main kernels: MFMA 16x16x32; tiles go HBM -> LDS directly (buffer_load_dwordx4 ... lds, no staging registers, no ds_write);
// bank conflicts are avoided by an XOR swizzle applied on the global-address side.  In the 8-wave kernel a K tile is consumed
// in four phases (k half x M half) of 16 MFMAs; the fragments of the next phase are read during the current one, the barrier
// that publishes the next stage sits in front of the last phase, and the loads of tile kt+2 are issued under that phase's
// MFMAs.  Long reductions run a 4-wave variant (128x128 wave tiles, one wave per SIMD; see w4_pays).
// K tails (K % 64 != 0: a weight gradient over an odd number of tokens, a forward over a width like 688): the lanes of the
// last K tile's loads that lie past K get an offset outside the buffer, which reads as zero; nothing else differs.  (A register-
// staged kernel used to cover them, without split last rounds and without the one-launch input gradient: a training step over
// 4 x 1000 tokens at h = 2048 took 4977 us with it and 4626 with these.)
// Blocks are renumbered so that each XCD (own L2) works on a contiguous band of tiles, 8 tiles tall.
//
// Tile counts that leave the last round of workgroups mostly empty (320 tiles on 256 CUs, or 64 tiles in all) are evened out
// by splitting the reduction of the tiles of that last round over several workgroups (given a workspace): each writes an
// fp32 partial tile and a small kernel adds the partials in a fixed order, so results stay bit-reproducible.
//
// Where that leaves fewer CUs idle the 4-wave kernel runs on tiles of 192 rows; products that do not fill the chip with either run on the smaller
// tiles of gemm_small.hip (see choose_plan).
#include "gemm_tile.h"
#include "gemm_list.h"

#include <math.h>

namespace {

template <typename OutT> __device__ __forceinline__ void store_out(OutT* p, float v, bool accumulate);
template <> __device__ __forceinline__ void store_out<bf16_t>(bf16_t* p, float v, bool accumulate) {
    *p = (bf16_t)(accumulate ? v + (float)*p : v);
}
template <> __device__ __forceinline__ void store_out<float>(float* p, float v, bool accumulate) {
    *p = accumulate ? v + *p : v;
}

// =================================================================================================
// main kernel: direct-to-LDS loads, XOR-swizzled tiles
// =================================================================================================
constexpr int DTILE = 256 * 64;  // elements per operand per stage of the swizzled layout (32 KiB)

// Work split of a launch: tile ids below `full` are one workgroup each; every later
// tile is computed by `nsplit` workgroups that each take a contiguous share of the K tiles and leave an fp32 partial tile.
struct SplitPlan {
    int full, rest, nsplit;  // rest: tiles - full
    float* partial;          // [rest][nsplit][tile]
};
// Split tile and share of workgroup-sized piece u >= full: like the whole tiles, an XCD's pieces are neighbours, all of one share where they can
// be (product in two shares, 1531 x 4096 x 11008, tile by tile 179 us, share by share 159; x 32000 403, 384).
__device__ __forceinline__ void split_piece(const SplitPlan& plan, int u, int& tile, int& part) {
    u -= plan.full;
    const int n = plan.rest * plan.nsplit, per = n >> 3, rem = n & 7, xcd = u & 7;
    u = xcd * per + (xcd < rem ? xcd : rem) + (u >> 3);
    part = u / plan.rest;
    tile = u - part * plan.rest;
}


#define SG_MFMA 0x008
#define SG_VMEM_R 0x020
#define SG_DS_R 0x100

// Instruction-scheduling recipe for one phase (compile-time unrolled): one MFMA, then up to PER LDS reads while reads are
// left, then up to PER_V global->LDS loads while loads are left.
template <int MASK, int N>
__device__ __forceinline__ void sched_group() {
    if constexpr (N > 0) __builtin_amdgcn_sched_group_barrier(MASK, N, 0);
}
template <int G, int NM, int RD, int PER, int NLD, int PER_V>
struct SchedPhase {
    static __device__ __forceinline__ void run() {
        if constexpr (G < NM) {
            sched_group<SG_MFMA, 1>();
            constexpr int left = RD - G * PER;
            constexpr int ds_slots = PER > 0 ? (RD + PER - 1) / PER : 0;
            constexpr int vleft = G >= ds_slots ? NLD - (G - ds_slots) * PER_V : 0;
            sched_group<SG_DS_R, (left > PER ? PER : (left > 0 ? left : 0))>();
            sched_group<SG_VMEM_R, (vleft > PER_V ? PER_V : (vleft > 0 ? vleft : 0))>();
            SchedPhase<G + 1, NM, RD, PER, NLD, PER_V>::run();
        }
    }
};

// 8 waves (2 x 4), each owning 128 x 64 of the 256 x 256 block tile as 8 x 4 MFMA 16x16x32 tiles.  The 16x16x32 shape is
// used because it sustains a higher clock than 32x32x16 under the board's power limit (fewer accumulator-register
// accesses per flop).  A 64-wide K tile is worked off in four phases (k half, M half): a phase issues 16 MFMAs on 4 A and
// 4 B fragments while the fragments of the next phase are read from LDS into the other register set.
//
template <bool A_KC, bool B_KC, typename OutT, bool MULTI, bool KTAIL>
__global__ __launch_bounds__(512) void gemm_d2l_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B, OutT* __restrict__ C,
                                                       int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int accumulate,
                                                       int tiles_m, int tiles_n, const SplitPlan plan, const KSegments seg) {
    constexpr int NW = 8, WAVES_N = 4;
    __shared__ __attribute__((aligned(1024))) bf16_t smem[4 * DTILE];  // A0 B0 A1 B1
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;

    int pid = blockIdx.x, part = 0;
    const bool split = pid >= plan.full;
    if (!split) {  // XCD-aware renumbering over the whole-tile workgroups
        const int per = plan.full >> 3, rem = plan.full & 7, xcd = pid & 7, idx = pid >> 3;
        pid = xcd * per + (xcd < rem ? xcd : rem) + idx;
    } else {
        split_piece(plan, pid, pid, part);
        pid += plan.full;
    }
    int tm, tn;
    tile_of(pid, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;

    TileLoader<A_KC, BM, NW, KTAIL> la;
    TileLoader<B_KC, BN, NW, KTAIL> lb;
    // per-lane offsets are 32-bit and relative to the block's first row / column (a scalar 64-bit advance of the operand
    // base), so operands of more than 2^31 elements are addressable
    const int64_t a_blk = A_KC ? (int64_t)m0 * lda : (int64_t)m0;
    const int64_t b_blk = B_KC ? (int64_t)n0 * ldb : (int64_t)n0;
    la.init(lane, wave, M - m0, lda);
    lb.init(lane, wave, N - n0, ldb);

    f32x4 acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

    int nk = MULTI ? seg.nk : (K + BK - 1) / BK, kt0 = 0;  // this workgroup's K tiles: kt0 .. kt0 + nk - 1
    if (split) {
        kt0 = (int)((int64_t)nk * part / plan.nsplit);
        nk = (int)((int64_t)nk * (part + 1) / plan.nsplit) - kt0;
    }
    const int64_t astep = A_KC ? BK : (int64_t)BK * lda;
    const int64_t bstep = B_KC ? BK : (int64_t)BK * ldb;
    const int arow = wm * 128, brow = wn * 64;

    bf16x8 fa[2][4], fb[2][4];
    auto read_a = [&](const bf16_t* sA, int ks, int half, int buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fa[buf][i] = sfrag<A_KC, 256>(sA, arow + half * 64 + i * 16, ks, lane);
    };
    auto read_b = [&](const bf16_t* sA, int ks, int buf) {
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[buf][j] = sfrag<B_KC, 256>(sA + DTILE, brow + j * 16, ks, lane);
    };
    // B is the first MFMA operand: the accumulator then holds C^T fragments, i.e. a lane owns 4 consecutive columns of one
    // row of C, which it can store as one vector.
    auto mfmas = [&](int half, int abuf, int bbuf) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[half * 4 + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[bbuf][j], fa[abuf][i], acc[half * 4 + i][j], 0, 0, 0);
    };
    auto issue_tile = [&](int t, int stage) {
        const bf16_t *Ab, *Bb;
        int kv;
        t += kt0;
        pick_segment<MULTI>(A, B, K, seg, t, kv, Ab, Bb);
        la.issue(la.base(Ab + a_blk + (int64_t)t * astep), smem + stage * 2 * DTILE, lane, wave, kv);
        lb.issue(lb.base(Bb + b_blk + (int64_t)t * bstep), smem + stage * 2 * DTILE + DTILE, lane, wave, kv);
    };

    issue_tile(0, 0);
    if (nk > 1) issue_tile(1, 1);
    // Pull the remaining kernel arguments into registers now: a scalar load still in flight inside the K loop shares the
    // counter of the LDS reads and would turn every counted wait on them into a full drain.
    asm volatile("" ::"s"(C), "s"(ldc), "s"(accumulate), "s"(plan.partial), "s"(plan.full), "s"(plan.nsplit));
    if constexpr (MULTI) asm volatile("" ::"s"(seg.A1), "s"(seg.B1), "s"(seg.A2), "s"(seg.B2), "s"(seg.t1), "s"(seg.t2), "s"(seg.K1), "s"(seg.K2));
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __syncthreads();
    read_b(smem, 0, 0);
    read_a(smem, 0, 0, 0);

    constexpr int RA = A_KC ? 4 : 8, RB = B_KC ? 4 : 8;  // LDS reads per fragment set
    constexpr int NM = 16;                                // MFMAs per phase
    constexpr int NLD = 2 * (32 / NW);                    // global->LDS loads per wave and tile pair
    // phases 0 and 2 fetch the A fragments of the other M half; phases 1 and 3 fetch B and A of the next k half
#define EZL_PHASE_SCHED(RD, LD) SchedPhase<0, NM, (RD), ((RD) + 11) / 12, (LD), 1>::run()
#define EZL_STEP(HAS_NEXT, DO_LOAD)                                                                       \
    {                                                                                                     \
        const int cur = kt & 1;                                                                           \
        const bf16_t* sA = smem + cur * 2 * DTILE;                                                         \
        read_a(sA, 0, 1, 1);                                                                              \
        mfmas(0, 0, 0);                                                                                   \
        EZL_PHASE_SCHED(RA, 0);                                                                           \
        read_b(sA, 1, 1);                                                                                 \
        read_a(sA, 1, 0, 0);                                                                              \
        mfmas(1, 1, 0);                                                                                   \
        EZL_PHASE_SCHED(RA + RB, 0);                                                                      \
        read_a(sA, 1, 1, 1);                                                                              \
        mfmas(0, 0, 1);                                                                                   \
        EZL_PHASE_SCHED(RA, 0);                                                                           \
        __builtin_amdgcn_sched_barrier(0);                                                                \
        __builtin_amdgcn_s_waitcnt(0x0F70);                                                               \
        __syncthreads();                                                                                  \
        __builtin_amdgcn_sched_barrier(0);                                                                \
        if (HAS_NEXT) {                                                                                   \
            read_b(smem + (cur ^ 1) * 2 * DTILE, 0, 0);                                                    \
            read_a(smem + (cur ^ 1) * 2 * DTILE, 0, 0, 0);                                                 \
        }                                                                                                 \
        if (DO_LOAD) issue_tile(kt + 2, cur);                                                             \
        mfmas(1, 1, 1);                                                                                   \
        EZL_PHASE_SCHED((HAS_NEXT) ? RA + RB : 0, (DO_LOAD) ? NLD : 0);                                   \
        __builtin_amdgcn_sched_barrier(0);                                                                \
    }

    int kt = 0;
    for (; kt + 2 < nk; ++kt) EZL_STEP(true, true)
    if (kt + 1 < nk) {
        EZL_STEP(true, false)
        ++kt;
    }
    EZL_STEP(false, false)
#undef EZL_STEP
#undef EZL_PHASE_SCHED

    if (split) {  // this workgroup's share of the reduction, as a dense fp32 tile; gemm_split_reduce_kernel adds the shares
        float* tile = plan.partial + ((size_t)(pid - plan.full) * plan.nsplit + part) * (size_t)(BM * BN);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *reinterpret_cast<f32x4*>(tile + (arow + i * 16 + (lane & 15)) * BN + brow + j * 16 + 4 * (lane >> 4)) = acc[i][j];
        return;
    }
    const int mrem = M - m0 < BM ? M - m0 : BM, nrem = N - n0;
    OutT* Ct = C + (int64_t)m0 * ldc + n0;
    if (N % 8 == 0 && ldc % (16 / (int)sizeof(OutT)) == 0 && ((uintptr_t)C & 15) == 0 && ldc < (1 << 21) / ((int)sizeof(OutT) / 2)) {
        store_tile_flags<8, 4, OutT, true, A_KC && B_KC>(acc, Ct, ldc, mrem, nrem, arow, brow, lane, accumulate);
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {  // any width, alignment and row stride: element by element
        const int row = arow + i * 16 + (lane & 15);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = brow + j * 16 + 4 * (lane >> 4);
            if (row >= mrem || col >= nrem) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (col + r < nrem)
                    store_out<OutT>(Ct + (int64_t)row * ldc + col + r, accumulate & kRoundResult ? (float)(bf16_t)acc[i][j][r] : acc[i][j][r],
                                    (accumulate & 1) != 0);
        }
    }
}


// =================================================================================================
// 4-wave form of the main kernel: 2 x 2 waves, each owning 128 x 128 of the block tile
// =================================================================================================
// One wave per SIMD with 8 x 8 MFMA 16x16x32 tiles: the 256 accumulator registers live in AGPRs, a K tile costs a third
// fewer LDS fragment reads than with 128 x 64 wave tiles, and nothing else runs on the SIMD to cover a stall, so the K loop
// is laid out step by step (one MFMA per step, a sched_barrier after each):
//   phase A of tile kt: 64 MFMAs on k half 0 (fragment set 0); the 16 fragments of k half 1 are read meanwhile and the 8 wave
//                       loads of B tile kt + 2 go out into the stage of B tile kt - 1
//   wait for A tile kt + 1 (B tile kt + 1 is older, B tile kt + 2 stays in flight) + barrier: tile kt + 1 has landed, every wave is
//                       done reading the stages of tile kt
//   phase B of tile kt: 64 MFMAs on k half 1 (set 1); the fragments of tile kt + 1, k half 0 are read meanwhile and the 8 wave
//                       loads of A tile kt + 2 go out into the stage of A tile kt
// What bounds it is the way of the operands' lines to the CU.  With two stages of both operands, all 16 loads in phase B and waited for
// behind the next phase A, operands from HBM (weights, in every step) cost as much with zeros in them, where no clock gives way, as with
// random data: loads alone took 1.45 us per K tile, from the last-level cache 1.0, the products 1.25.  The 160 KiB hold two stages
// of A and three of B, loads go out in the first half of each phase (one every fourth MFMA: the CU's address unit takes 16 cycles per 1 KiB wave
// load, the four waves' keep it busy for just that half; every second MFMA 99 us where this takes 96, B's over all of phase A 97), and B
// has more than a K tile's time on the way, A three quarters.  Operands from HBM, us before and now: 4096 x 4096 x 4096 109 -> 96,
// 4096 x 4096 x 11008 277 -> 240, 2048 x 4096 x 11008 271 -> 206, weight gradient 11008 x 4096 x 4096 314 -> 288; from the cache 94 -> 94, 233 -> 230.
// The loop's back edge sits right behind the barrier, where no LDS read is in flight, so inside the body the compiler's
// waits on the fragment reads are exact counts.  Reads are issued in the first half of a phase (one every second MFMA) and
// have landed long before the next phase needs them.
// A workgroup works off items blockIdx.x, + gridDim.x, ... as one stream of K tiles: the last K tiles of an item bring in the
// first two of the next, and the finished accumulators are stored while those are on their way (their wait is a count that
// leaves the stores in flight).  With one workgroup per tile a tile cost 14 us on top of its K tiles - a workgroup's start, the first
// loads, the stores drained before its LDS is free - which is a third of it at 32 K tiles: 4000 x 32000 x 2048 444 -> 407 us,
// 8192 x 32000 x 1024 517 -> 460, 4096 x 11008 x 2048 143 -> 134, 8192 x 32000 x 5120 1974 -> 1947; the weight gradient 32000 x 4096 x
// 4096 911 -> 885.  What is left there is the power limit: longer K loops run at 1.2 - 1.35 us per K tile instead of 0.96.
// TBM = 192: six tiles of 16 rows per wave, 144 KiB, for products whose 256 x 256 tiles leave more CUs idle (see kRates).
// C must allow 16-byte stores (N and ldc multiples of 8 for bf16, of 4 for fp32, aligned base), its tile-relative byte offsets
// must fit 31 bits, and every item must have two K tiles or more: the host side checks.
// LIST (forward, weight gradients): the tiles of several products over one K; what is said per product comes from the list then, not from the
// other arguments.  A decoder layer's seven weight gradients over 4000 tokens (h = 2048, f = 5504: 784 tiles, three rounds and 16 tiles) went out
// as 128 x 128 tiles in 453 us, as these in 387; its gate and up products (704 tiles) as 256 x 128 tiles in 208, as these in 155.  (One
// product in a list of one would save the form without it, but costs 6 us a launch: a tile's scalar loads depend on one another.)
struct NoList {};
template <bool A_KC, bool B_KC, typename OutT, bool MULTI, bool KTAIL, bool LIST = false, int TBM = 256>
__global__ __launch_bounds__(256, 1) void gemm_w4_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B, OutT* __restrict__ C,
                                                         int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int accumulate,
                                                         int tiles_m, int tiles_n, int items, const SplitPlan plan, const KSegments seg,
                                                         const std::conditional_t<LIST, GemmSmallArgs, NoList> list) {
    static_assert(!LIST || (A_KC == B_KC && !MULTI), "lists are of forward products or weight gradients");
    constexpr int TM = TBM / 32, NA = TM, NB = 8;  // MFMA tiles of a wave, one below the other; wave loads of an A and a B tile
    constexpr int ASTAGE = TBM * BK;
    __shared__ __attribute__((aligned(1024))) bf16_t smem[2 * ASTAGE + 3 * DTILE];  // A0 A1 B0 B1 B2
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int nk_all = MULTI ? seg.nk : (K + BK - 1) / BK;
    const int64_t astep = A_KC ? BK : (int64_t)BK * lda;
    const int64_t bstep = B_KC ? BK : (int64_t)BK * ldb;
    const int arow = wm * (TBM / 2), brow = wn * 128;

    struct ListItem {  // its product, its operands from the tile's corner on, their strides, the tile's rows and columns
        int product, lda, ldb, mrem, nrem;
        const bf16_t *a, *b;
    };
    struct Item : std::conditional_t<LIST, ListItem, NoList> {  // a whole tile, or a tile of the split last round with this workgroup's share of its K tiles
        int m0, n0, kt0, nk;
        int slot;  // >= 0: place of the partial tile
        int64_t a_blk, b_blk;
    };
    auto item_of = [&](int u) {
        Item it;
        it.kt0 = 0; it.nk = nk_all; it.slot = -1;
        int pid = u;
        if (u < plan.full) {  // XCD-aware renumbering over the whole tiles (a grid smaller than the items is a multiple of 8)
            const int per = plan.full >> 3, rem = plan.full & 7, xcd = u & 7, idx = u >> 3;
            pid = xcd * per + (xcd < rem ? xcd : rem) + idx;
        } else {
            int t, part;
            split_piece(plan, u, t, part);
            it.slot = t * plan.nsplit + part;
            pid = plan.full + t;
            it.kt0 = (int)((int64_t)nk_all * part / plan.nsplit);
            it.nk = (int)((int64_t)nk_all * (part + 1) / plan.nsplit) - it.kt0;
        }
        int tm, tn;
        if constexpr (LIST) {
            pid = __builtin_amdgcn_readfirstlane(pid);
            it.product = 0;
#pragma unroll
            for (int j = 1; j < kMaxProblems; ++j) it.product += pid >= list.first[j];
            const GemmProblem& p = list.p[it.product];
            tile_of(pid - p.first, p.tiles_m, p.tiles_n, tm, tn);
        } else {
            tile_of(pid, tiles_m, tiles_n, tm, tn);
        }
        // (scalar registers: the buffer bases are made of them)
        it.m0 = __builtin_amdgcn_readfirstlane(tm * TBM);
        it.n0 = __builtin_amdgcn_readfirstlane(tn * BN);
        it.kt0 = __builtin_amdgcn_readfirstlane(it.kt0);
        it.nk = __builtin_amdgcn_readfirstlane(it.nk);
        it.slot = __builtin_amdgcn_readfirstlane(it.slot);
        it.a_blk = A_KC ? (int64_t)it.m0 * lda : (int64_t)it.m0;
        it.b_blk = B_KC ? (int64_t)it.n0 * ldb : (int64_t)it.n0;
        if constexpr (LIST) {
            const GemmProblem& p = list.p[it.product];
            it.a = p.A + (A_KC ? it.m0 * p.lda : it.m0);
            it.b = p.B + (B_KC ? it.n0 * p.ldb : it.n0);
            it.lda = (int)p.lda;
            it.ldb = (int)p.ldb;
            it.mrem = min(p.M - it.m0, TBM);
            it.nrem = min(p.N - it.n0, BN);
            // (these scalar loads are waited for here, not inside the K loop)
            asm volatile("" ::"s"(it.a), "s"(it.b), "s"(it.lda), "s"(it.ldb), "s"(it.mrem), "s"(it.nrem));
        }
        return it;
    };
    auto rows_left = [&](const Item& x) {
        if constexpr (LIST) return x.mrem;
        else return M - x.m0;
    };
    auto cols_left = [&](const Item& x) {
        if constexpr (LIST) return x.nrem;
        else return N - x.n0;
    };
    auto a_stride = [&](const Item& x) {
        if constexpr (LIST) return (int64_t)x.lda;
        else return lda;
    };
    auto b_stride = [&](const Item& x) {
        if constexpr (LIST) return (int64_t)x.ldb;
        else return ldb;
    };
    if constexpr (LIST) {  // every cache line of the list, fetched at once: the loads below depend on one another
        int line[kMaxProblems];
#pragma unroll
        for (int j = 0; j < kMaxProblems; ++j) line[j] = list.p[j].M;
        asm volatile("" ::"s"(line[0]), "s"(line[1]), "s"(line[2]), "s"(line[3]), "s"(line[4]), "s"(line[5]), "s"(line[6]), "s"(list.first[6]));
    }
    int u = blockIdx.x;
    Item it = item_of(u);

    TileLoader<A_KC, TBM, 4, KTAIL> la;
    TileLoader<B_KC, BN, 4, KTAIL> lb;
    la.init(lane, wave, rows_left(it), a_stride(it));
    lb.init(lane, wave, cols_left(it), b_stride(it));

    FragReader<A_KC, TBM> ra;
    FragReader<B_KC, BN> rb;
    ra.init(arow, lane);
    rb.init(brow, lane);

    f32x4 acc[TM][8];
    bf16x8 fa[2][TM], fb[2][8];
    // fragment f of a k half: f < 8 the B fragment f, else the A fragment f - 8
    auto read_frag = [&](const bf16_t* sA, const bf16_t* sB, int ks, int buf, auto F) {
        constexpr int f = decltype(F)::value;
        if constexpr (f < 8) fb[buf][f] = rb.template read<f>(sB, ks);
        else fa[buf][f - 8] = ra.template read<f - 8>(sA, ks);
    };
    __amdgpu_buffer_rsrc_t ga, gb;
    int kva = BK, kvb = BK;
    auto a_base = [&](const Item& x, int t) {
        t += x.kt0;
        if constexpr (LIST) {
            kva = K - t * BK;
            ga = la.base(x.a + (int64_t)t * BK * (A_KC ? 1 : x.lda));
        } else {
            const bf16_t *Ab, *Bb;
            pick_segment<MULTI>(A, B, K, seg, t, kva, Ab, Bb);
            ga = la.base(Ab + x.a_blk + (int64_t)t * astep);
        }
    };
    auto b_base = [&](const Item& x, int t) {
        t += x.kt0;
        if constexpr (LIST) {
            kvb = K - t * BK;
            gb = lb.base(x.b + (int64_t)t * BK * (B_KC ? 1 : x.ldb));
        } else {
            const bf16_t *Ab, *Bb;
            pick_segment<MULTI>(A, B, K, seg, t, kvb, Ab, Bb);
            gb = lb.base(Bb + x.b_blk + (int64_t)t * bstep);
        }
    };
    // load l of a tile pair: l < NA piece l of the A tile, else of the B tile
    auto issue_load = [&](bf16_t* sA, bf16_t* sB, auto L) {
        constexpr int l = decltype(L)::value;
        if constexpr (l < NA) la.template issue_at<l>(ga, sA, lane, wave, kva);
        else lb.template issue_at<l - NA>(gb, sB, lane, wave, kvb);
    };

    int a0 = 0, a1 = ASTAGE, b0 = 2 * ASTAGE, b1 = b0 + DTILE, b2 = b1 + DTILE;  // stages of K tiles kt, kt + 1 (and kt + 2)
    a_base(it, 0);
    b_base(it, 0);
    static_for<0, NA + NB>([&](auto L) { issue_load(smem + a0, smem + b0, L); });
    a_base(it, 1);
    b_base(it, 1);
    static_for<0, NA + NB>([&](auto L) { issue_load(smem + a1, smem + b1, L); });
    // the remaining kernel arguments, pulled into registers now (a scalar load in flight inside the K loop would share the
    // counter of the LDS reads)
    asm volatile("" ::"s"(C), "s"(ldc), "s"(accumulate), "s"(plan.partial), "s"(plan.full), "s"(plan.nsplit), "s"(items), "s"(M), "s"(N),
                 "s"(tiles_m), "s"(tiles_n));
    if constexpr (MULTI) asm volatile("" ::"s"(seg.A1), "s"(seg.B1), "s"(seg.A2), "s"(seg.B2), "s"(seg.t1), "s"(seg.t2), "s"(seg.K1), "s"(seg.K2));
    static_assert(NA + NB <= 16, "a count's low bits, and bit 4 alone");
    __builtin_amdgcn_s_waitcnt(NA + NB == 16 ? 0x4070 : 0x0070 | (NA + NB));  // lgkmcnt(0): K tile 0 has landed, K tile 1 is still on its way
    wave_barrier();
    static_for<0, TM + 8>([&](auto F) { read_frag(smem + a0, smem + b0, 0, 0, F); });

    constexpr int RSTEP = 2;  // a fragment read every RSTEP MFMAs (of 8 x 8 MFMA tiles 16 reads: the first half of a phase)
    constexpr int LSTEP = 4;  // a tile load every LSTEP MFMAs (8 loads: the first half of a phase)
    auto phase_a = [&](const bf16_t* sA, const bf16_t* sB, bf16_t* lB) {
        static_for<0, TM * 8>([&](auto S) {
            constexpr int m = decltype(S)::value, i = m >> 3, j = m & 7;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[0][j], fa[0][i], acc[i][j], 0, 0, 0);
            if constexpr (m % RSTEP == 0 && m / RSTEP < TM + 8) read_frag(sA, sB, 1, 1, std::integral_constant<int, m / RSTEP>{});
            if constexpr (m % LSTEP == LSTEP - 1 && m / LSTEP < NB) issue_load(smem, lB, std::integral_constant<int, NA + m / LSTEP>{});
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto phase_b = [&](const bf16_t* sA, const bf16_t* sB, bf16_t* lA) {
        static_for<0, TM * 8>([&](auto S) {
            constexpr int m = decltype(S)::value, i = m >> 3, j = m & 7;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[1][j], fa[1][i], acc[i][j], 0, 0, 0);
            if constexpr (m % RSTEP == 0 && m / RSTEP < TM + 8) read_frag(sA, sB, 0, 0, std::integral_constant<int, m / RSTEP>{});
            if constexpr (m % LSTEP == LSTEP - 1 && m / LSTEP < NA) issue_load(lA, smem, std::integral_constant<int, m / LSTEP>{});
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto publish = [&](auto LEFT) {  // all but this wave's LEFT newest accesses are done: the next K tile has landed; so are its LDS reads
        constexpr int left = decltype(LEFT)::value;
        __builtin_amdgcn_s_waitcnt(0x0070 | (left & 15) | ((left >> 4) << 14));
        wave_barrier();
    };
    // newer than the A tile that is waited for: the B tile behind the next, and where an item begins the stores of the one before (a count
    // holds at most 63)
    typedef std::integral_constant<int, NB> ahead;
    constexpr int STORES = TM * 8 * (int)sizeof(OutT) / 4;
    typedef std::integral_constant<int, NB + STORES <= 63 ? NB + STORES : 63> ahead_and_stores;
    auto flip = [&]() {
        const int x = a0, y = b0;
        a0 = a1;
        a1 = x;
        b0 = b1;
        b1 = b2;
        b2 = y;
        asm volatile("" : "+s"(a0), "+s"(a1), "+s"(b0), "+s"(b1), "+s"(b2));  // (the fragment reads are restrict-qualified: a refilled stage must not look like the same address)
    };
    // the next A and B tile to bring in: K tile ta (tb) of item ia (ib)
    Item ia = it, ib = it;
    int ta = 2, tb = 2;
    auto advance_a = [&](const Item& next) __attribute__((always_inline)) {
        if (ta == ia.nk) {
            if (min(rows_left(next), TBM) != min(rows_left(ia), TBM) || (LIST && a_stride(next) != a_stride(ia))) la.init(lane, wave, rows_left(next), a_stride(next));
            ia = next;
            ta = 0;
        }
        a_base(ia, ta++);
    };
    auto advance_b = [&](const Item& next) __attribute__((always_inline)) {
        if (tb == ib.nk) {
            if (min(cols_left(next), BN) != min(cols_left(ib), BN) || (LIST && b_stride(next) != b_stride(ib))) lb.init(lane, wave, cols_left(next), b_stride(next));
            ib = next;
            tb = 0;
        }
        b_base(ib, tb++);
    };
    for (bool first = true;; first = false) {
        const int next_u = u + (int)gridDim.x;
        const bool more = next_u < items;
        const Item next = more ? item_of(next_u) : it;  // (behind the last item its own first tiles again, into stages nobody reads)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        advance_b(next);
        phase_a(smem + a0, smem + b0, smem + b2);
        if (first) publish(ahead{});
        else publish(ahead_and_stores{});
        for (int left = it.nk - 1; left > 0; --left) {
            advance_a(next);
            phase_b(smem + a1, smem + b1, smem + a0);
            advance_b(next);
            phase_a(smem + a1, smem + b1, smem + b0);
            publish(ahead{});
            flip();
        }
        advance_a(next);
        phase_b(smem + a1, smem + b1, smem + a0);
        flip();
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(acc[i][j]));
        int64_t ld = ldc;
        asm volatile("" : "+s"(ld));  // (the stores' offsets are not kept over the K loop)
        if (it.slot >= 0) {  // a share of the reduction, as a dense fp32 tile; gemm_split_reduce_kernel adds the shares
            float* tile = plan.partial + (size_t)it.slot * (size_t)(TBM * BN);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    *reinterpret_cast<f32x4*>(tile + (arow + i * 16 + (lane & 15)) * BN + brow + j * 16 + 4 * (lane >> 4)) = from_agprs<TM * 8>(acc[i][j]);
        } else if constexpr (LIST) {
            const GemmProblem& p = list.p[it.product];
            OutT* Ct = (OutT*)p.C + (int64_t)it.m0 * p.ldc + it.n0;
            store_tile_flags<TM, 8, OutT, true, false>(acc, Ct, p.ldc, it.mrem, it.nrem, arow, brow, lane, p.accumulate);
        } else {
            const int mrem = M - it.m0 < TBM ? M - it.m0 : TBM;
            OutT* Ct = C + (int64_t)it.m0 * ld + it.n0;
            store_tile_flags<TM, 8, OutT, true, A_KC && B_KC>(acc, Ct, ld, mrem, N - it.n0, arow, brow, lane, accumulate);
        }
        if (!more) break;
        it = next;
        u = next_u;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the last item's loads of a next tile (its own again) may not outlive the workgroup's LDS
}

// Sum in index order of the vectors at src, src + stride, ...: `count` partial results, read once, up to eight at a time.
__device__ __forceinline__ f32x4 sum_partials(const float* __restrict__ src, size_t stride, int count) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    const auto add = [&](auto COUNT) {
        constexpr int n = decltype(COUNT)::value;
        for (; count >= n; count -= n, src += n * stride) {
            f32x4 x[n];
#pragma unroll
            for (int p = 0; p < n; ++p) x[p] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(src + p * stride));
#pragma unroll
            for (int p = 0; p < n; ++p)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += x[p][e];
        }
    };
    add(std::integral_constant<int, 8>{});
    add(std::integral_constant<int, 4>{});
    add(std::integral_constant<int, 2>{});
    add(std::integral_constant<int, 1>{});
    return v;
}

// C tile (=|+=) sum of the nsplit fp32 partial tiles, added in index order.  A wave owns a row of a tile, a lane four consecutive columns
// of it.  What bounds it is the read of the partial tiles, which comes from the last-level cache mostly: every load instruction is 1 KiB of one row, and
// up to eight of a lane's are in flight.  (With 16 consecutive columns a thread, whose loads of a wave lay 64 bytes apart, and a part at a time, us before and now, M x N of a
// product, tiles x shares: 1531 x 4096, 128 of 192 rows x 2 16.3 -> 10.2; 2048 x 768, 24 x 10 18.0 -> 10.4; 1167 x 1024, 20 x 12 17.1 -> 9.3; 4000 x 2048, 128 x 2
// 22.3 -> 12.8; fp32, 50304 x 1024, 20 x 2 5.8 -> 4.6.)
constexpr int kReduceRows = 4;  // rows of a block
template <typename OutT, int TBM>
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(OutT* __restrict__ C, int M, int N, int64_t ldc, int accumulate,
                                                                int tiles_m, int tiles_n, const SplitPlan plan) {
    constexpr int PIECES = TBM / kReduceRows;
    const int t = blockIdx.x / PIECES;  // split tile
    int tm, tn;
    tile_of(plan.full + t, tiles_m, tiles_n, tm, tn);
    const int rl = (blockIdx.x - t * PIECES) * kReduceRows + (threadIdx.x >> 6), cl = (threadIdx.x & 63) * 4;
    const int row = tm * TBM + rl, col = tn * BN + cl;
    if (row >= M || col >= N) return;
    f32x4 v = sum_partials(plan.partial + (size_t)t * plan.nsplit * (TBM * BN) + (size_t)rl * BN + cl, TBM * BN, plan.nsplit);
    if (accumulate & kRoundResult) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (float)(bf16_t)v[e];
        accumulate &= 1;
    }
    OutT* dst = C + (int64_t)row * ldc + col;
    if (col + 4 <= N && ldc % 8 == 0 && ((uintptr_t)C & 15) == 0) {
        typedef OutT vec_t __attribute__((ext_vector_type(4)));
        vec_t o;
        if (accumulate) {
            const vec_t old = *reinterpret_cast<const vec_t*>(dst);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (OutT)(v[e] + (float)old[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (OutT)v[e];
        }
        *reinterpret_cast<vec_t*>(dst) = o;
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (col + e < N) store_out<OutT>(dst + e, v[e], accumulate != 0);
}

enum Class { kForward, kInputGradient, kWeightGradient };
// Products whose widths are whole cache lines (128 bytes): what the rates, the 192 x 256 tiles and the wider rule for split rounds below were
// measured on.  Other widths, and weight gradients over up to 16 K tiles, which are bound by their results, keep the rates that were fitted to all widths.
// Only the widths are looked at, not how the rows lie: rows of a whole width that straddle lines (a column slice, a pitch of 8 elements more, a base 16 bytes off) cost up to 30 %
// more on any tile (4096 x 4096 x 4096 103 us with such an A, 111 with both, 120 with both bases off), and the plans for whole lines are the better ones there too: of
// 156 such products 5 - 8 % (forward), 5 - 9 % (input gradients) and 2 % (weight gradients) faster than with the rates for other widths.
bool whole_lines(Class cls, int64_t M, int64_t N, int64_t K) {
    return N % 64 == 0 && (cls == kWeightGradient ? M % 64 == 0 && K > 16 * BK : K % 64 == 0);
}

// Split the tiles of a mostly empty last round?  cus workgroups run at a time (one per CU: the kernels use 128 KiB of LDS and more).
constexpr int kCus = 256;
int64_t tile_bytes(int kind) { return gemm_kind_bm(kind) * gemm_kind_bn(kind) * (int64_t)sizeof(float); }
SplitPlan make_plan(int kind, bool lines, int64_t tiles, int64_t nk, void* workspace, int64_t workspace_bytes) {
    SplitPlan p;
    p.full = (int)tiles; p.rest = 0; p.nsplit = 1; p.partial = nullptr;
    const int64_t r = tiles % kCus;
    // Up to 96 tiles always: two shares and more of them.  97 - 128 are half a chip's worth, in two shares; time of them split over whole, 1400 products,
    // by K tiles 16 - 31 1.36, 32 - 47 1.07, 48 - 63 0.93, 96 - 127 0.75, 256 - 399 0.63 (behind whole rounds 1.12, 1.03, 0.98, 0.91, 0.82).
    if (r == 0 || r > (lines && nk >= 48 ? kCus / 2 : 96)) return p;
    const int s = (int)(kCus / r < nk / 8 ? kCus / r : nk / 8);  // a share of fewer than 8 K tiles is mostly prologue
    if (s < 2) return p;
    if (!workspace || workspace_bytes < r * s * tile_bytes(kind)) return p;
    p.full = (int)(tiles - r); p.rest = (int)r; p.nsplit = s; p.partial = (float*)workspace;
    return p;
}
int64_t split_bytes(int kind, bool lines, int64_t tiles, int64_t nk) {
    const SplitPlan p = make_plan(kind, lines, tiles, nk, (void*)16, INT64_MAX);
    return p.nsplit > 1 ? p.rest * p.nsplit * tile_bytes(kind) : 0;
}

// ---- which tile shape, and over how many workgroups a tile's reduction is split ------------------------------------------
// The time of a launch is estimated for every shape as first + rounds x (K tiles x rate + next) + out x MB of results and the cheapest one taken: us per
// 64-wide K tile of one workgroup per CU (two sharing a CU for 128 and 64 tiles), `low` with the chip nearly empty, `high` full, in between by a
// power of the share of it that is filled; the two ends of a round, and what the launch and its results cost.  Fits to 6000 products of 64 - 96000 wide
// operands, 100 - 16384 rows and 2 - 1100 K tiles, weights from HBM, each timed with every shape and several splits in changing order: what is
// taken is 1.0 % (forward, input gradients) and 0.9 % (weight gradients) slower than the fastest, and was 2.0 and 4.5 % with rates fitted to
// products alone on the chip, out of its caches (kOtherRates; still those of rows that are not whole lines and of lists).  M x N x K, us for
// 256 x 256 (the better of whole and split), 192 x 256, 256 x 128, 192 x 128, 128 x 128:
//   forward          1774 x 4096 x 3584 68, 59, 51, 76, 57        1556 x 3520 x 10752 123, 111, 124, 111, 148    3664 x 2368 x 2048 45, 38, 57, 47, 54
//   input gradient   1636 x 3840 x 30464 317, 445, 387, 483, 429  3033 x 1856 x 34432 374, 316, 456, 355, 469    4193 x 10048 x 4224 272, 277, 346, 330, 371
//   weight gradient  4032 x 3712 x 1664 51, 69, 67, 75, 68        1856 x 2176 x 4096 64, 60, 61, 51, 51          4480 x 5760 x 4160 194, 195, 234, 237, 235
// Without the 192 x 256 tiles the best of the others is 2.0 % slower in the mean, 3 % and more for every sixth product.  What makes the large tiles win is
// LDS traffic: a K tile of 256 x 128 (192 x 128) takes the LDS 1152 (960) cycles of 128 bytes, written and read, and its MFMAs 1024 (768); 192 x 256
// 1344 and 1536, 256 x 256 1536 and 2048.
// A split reduction adds a launch and a trip of the fp32 partial tiles through the caches (2048 x 768 x 4096 as 256 x 128 tiles
// split four ways: 26, of which 10 for that).
struct Rates {
    double low, high, first, next, power, out;
};
constexpr Rates kRates[3][kGemmKinds] = {
    {{0.904, 1.35, 5.789, 4.753, 1.329, 0.003}, {0.735, 1.058, 4.794, 3.77, 1.19, 0.011}, {0.68, 0.822, 3.52, 2.587, 2.252, 0.182}, {0.457, 0.67, 3.006, 2.612, 0.739, 0.137}, {0.56, 0.93, 2.444, 1.883, 2.136, 0.119}, {0.286, 0.405, 2.848, 0.321, 6, 0.466}, {0.096, 0.205, 2.107, 2.546, 0.3, 0.183}},
    {{0.986, 1.397, 6.138, 4.844, 1.422, 0}, {0.824, 1.098, 5.446, 3.786, 1.472, 0.01}, {0.713, 0.833, 3.462, 2.866, 2.656, 0.187}, {0.5, 0.66, 2.704, 3.02, 0.992, 0.143}, {0.637, 0.943, 3.112, 1.208, 4.766, 0.184}, {0.307, 0.464, 2.735, 0.783, 6, 0.372}, {0.115, 0.203, 2.294, 2.438, 0.3, 0.259}},
    {{1.088, 1.404, 7.566, 6.16, 1.4, 0.063}, {0.909, 1.098, 7.463, 3.783, 1.767, 0.087}, {0.665, 0.815, 5.6, 2.887, 0.602, 0.184}, {0.426, 0.669, 3.605, 2.771, 0.3, 0.189}, {0.553, 0.931, 2.861, 2.219, 1.454, 0.16}, {0.276, 0.457, 3.539, 0.1, 6, 0.263}, {0.148, 0.228, 2.623, 2.118, 0.3, 0.309}}};
constexpr Rates kOtherRates[2][kGemmKinds] = {
    {{0.72, 1.3, 0, 8.8, 1, 0}, {}, {0.57, 0.71, 0, 6.5, 3, 0}, {0.54, 0.57, 0, 5.4, 3, 0}, {0.69, 0.94, 0, 3.25, 99, 0}, {0.275, 0.43, 0, 2.6, 99, 0}, {0.187, 0.2, 0, 3.3, 3, 0}},
    {{1.18, 1.3, 0, 12.5, 1, 0}, {}, {0.74, 0.83, 0, 8, 3, 0}, {0.61, 0.695, 0, 6, 3, 0}, {0.64, 0.8, 0, 5, 99, 0}, {0.265, 0.45, 0, 2.7, 99, 0}, {0.21, 0.218, 0, 3.1, 3, 0}}};
// The partial tiles of 256 and 192 x 256 are added faster (gemm_split_reduce_kernel): 11 MB/us is the rate between 8 and 18 with the least loss over 80
// products whose plan it decides, 2.1 % faster in the mean than with 8, at worst 2.4 % slower.  Of 20000 other products it changes the plan of 640; 110 of those are 5.8 % faster
// in the mean, 18 slower by 1 - 7 % and one by 16 (14933 x 256 x 5504).  M x N x K, us with tiles x shares as with 8 and now: input gradient 3175 x 512 x
// 12224 82.8 (128 x 128, 5), 63.3 (192 x 256, 7); 5751 x 896 x 11776 169 (192 x 128), 138 (192 x 256, 2); forward 1743 x 1280 x 6528 53.7 (256 x 128, 3), 49.1 (192 x 256,
// 5); weight gradient 3072 x 1152 x 8485 94.5 (256 x 128, 2), 79.5 (192 x 256, 3).
constexpr double kReduceFixed = 4.0, kReduceBytesPerUs = 8e6, kLargeReduceBytesPerUs = 11e6;
double reduce_cost(int64_t tiles, int64_t tile_elems, int64_t nsplit, double bytes_per_us = kReduceBytesPerUs) {
    return kReduceFixed + (double)tiles * tile_elems * nsplit * 8 / bytes_per_us;
}
// What share of the way from `low` to `high` the rate goes with `groups` of kCus workgroups on the chip, of kRates' three rows and kOtherRates' two: the powers
// would be most of a search.
double way_up(int row, int kind, int64_t groups) {
    static const auto table = [] {
        static double t[5][kGemmKinds][kCus + 1];
        for (int r = 0; r < 5; ++r)
            for (int k = 0; k < kGemmKinds; ++k)
                for (int g = 0; g <= kCus; ++g) t[r][k][g] = pow((double)g / kCus, (r < 3 ? kRates[r] : kOtherRates[r - 3])[k].power);
        return &t;
    }();
    return (*table)[row][kind][groups];
}
// us of a launch of `tiles` tiles, results of out_mb MB
double cost_large(const Rates& rate, int row, int kind, bool lines, int64_t tiles, int64_t nk, int64_t room, double out_mb) {
    const SplitPlan p = make_plan(kind, lines, tiles, nk, (void*)16, room);
    auto round = [&](int64_t groups, int64_t k) { return k * (rate.low + (rate.high - rate.low) * way_up(row, kind, groups)) + rate.next; };
    double t = rate.first + rate.out * out_mb + (p.full / kCus) * (nk * rate.high + rate.next);
    if (p.full % kCus) t += round(p.full % kCus, nk);
    if (p.nsplit > 1) t += round(p.rest * p.nsplit, (nk + p.nsplit - 1) / p.nsplit) + reduce_cost(p.rest, tile_bytes(kind) / 4, p.nsplit, lines ? kLargeReduceBytesPerUs : kReduceBytesPerUs);
    return t;
}
double cost_small(const Rates& rate, int row, int kind, int64_t tiles, int64_t nk, int64_t nsplit, double out_mb) {
    const int64_t groups = tiles * nsplit, share = (nk + nsplit - 1) / nsplit;
    const bool two = kind == kTile128 || kind == kTile64;  // workgroups per CU
    const int64_t slots = two ? 2 * kCus : kCus, rest = groups % slots;
    double t = rate.first + rate.out * out_mb + (groups / slots) * (share * rate.high + rate.next);
    if (rest) t += share * (rate.low + (rate.high - rate.low) * way_up(row, kind, rest < kCus ? rest : kCus)) + rate.next;
    if (nsplit > 1) t += reduce_cost(tiles, gemm_kind_bm(kind) * gemm_kind_bn(kind), nsplit);
    return t;
}

int64_t tiles_of(int kind, int64_t M, int64_t N) {
    const int64_t bm = gemm_kind_bm(kind), bn = gemm_kind_bn(kind);
    return ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
}
// A list on 256 x 256 tiles has to win by a fourteenth: its tiles cost a chain of scalar loads each, and many rounds of short reductions are
// bound by the results' way to memory, whatever the launches.  Forward and backward of a layer with its weight gradients in such a list
// against without, by estimated ratio of the weight gradients (T, h, kv heads, f; us):
//   0.76 - 0.80   8192, 2048, 16, 5504 3867 -> 3680; 4000, 2048, 16, 5504 1905 -> 1835; 10086, 1024, 8, 3328 2471 -> 2432
//   0.80 - 0.93   4810, 2560, 20, 7744 3443 -> 3313; 1691, 2944, 23, 9216 1667 -> 1631; 2048, 4096, 8, 14336 2900 -> 2860; 2780, 2688, 21, 9408
//                 2283 -> 2205; at worst 2963, 1024, 2, 3392 707 -> 716
//   0.93 - 1.00   (before the margin) 1531, 4096, 32, 11008 2180 -> 2216; 8569, 896, 14, 2976 1772 -> 1787; 1331, 3200, 25, 9984 1589 -> 1550
// Gate and up in a forward list, by the same margin: 1726, 3072, 24, 9920 1760 -> 1709; 4952, 1792, 14, 4800 1968 -> 1923; 4000, 2048, 16, 5504
// 1748 -> 1716; 24 random layers 0.7 % faster in the mean, none slower.  (All of these, and kMargin256's below, with the 4-wave kernel's first form and against separate launches
// on kOtherRates' plans, by which the two are still compared.  Separate launches of whole lines that fill the chip have become 5 - 18 % faster since, so the decision leans to lists.)  bf16 weight gradients, whether list or single: 5183, 2048, 16, 6912 2641 -> 2526;
// 2961, 2048, 4, 5504 1288 -> 1231; 24 random layers 1.7 %, none slower.
constexpr double kMarginList256 = 0.93;
// `count` products over the same nk K tiles in one launch; `room`: workspace bytes.  256 x 256 tiles take one product, or with list_256 all
GemmPlan find_plan(Class cls, bool lines, int count, const int64_t* M, const int64_t* N, int64_t nk, int64_t room, double* time = nullptr, bool list_256 = false) {
    const bool wgrad = cls == kWeightGradient;
    const Rates* rates = lines ? kRates[cls] : kOtherRates[wgrad];
    const int row = lines ? cls : 3 + wgrad;
    double out_mb = 0;
    for (int i = 0; i < count; ++i) out_mb += (double)M[i] * N[i] * (wgrad ? 4e-6 : 2e-6);
    // 128 x 128 tiles read every operand most often, which lists of weight gradients over many tokens feel: a layer's seven over 11918 tokens at
    // h = 1024 400 us (estimate 309), with 256 x 128 tiles 354 (315).
    const double list_128 = wgrad && count > 3 ? 1.05 : 1;
    // Weight gradients of two rounds of 256 x 256 tiles or more, as of a vocabulary, are bound by their results' way to memory as much as by the tiles,
    // which the rates of one round do not know: the smaller tiles have to win by a twelfth.  50304 x 1024 x 1167, 256 x 256 against 128 x 128 tiles: 147, 175 us
    // (bf16 122, 131); bf16 70528 x 2176 x 477 198, 221; 151808 x 1024 x 711 299, 319.  160 such products: what is taken is 2.2 % behind the fastest, without
    // this 3.3 (those that overwrite fp32 2.9 and 5.4).
    double margin = 1;
    GemmPlan best = {kTile256, 1};
    double t_best = 1e30;
    if (count == 1 || list_256) {
        int64_t tiles = 0;
        for (int i = 0; i < count; ++i) tiles += tiles_of(kTile256, M[i], N[i]);
        if (wgrad && count == 1 && tiles >= 2 * kCus) margin = 1.08;
        t_best = cost_large(rates[kTile256], row, kTile256, lines, tiles, nk, room, out_mb) / (list_256 ? kMarginList256 : 1);
    }
    if (count == 1 && lines) {  // (no rates for others)
        const double t = cost_large(rates[kTile192x256], row, kTile192x256, lines, tiles_of(kTile192x256, M[0], N[0]), nk, room, out_mb);
        if (t * margin < t_best && nk >= 2) {
            t_best = t * margin;
            best.kind = kTile192x256;
        }
    }
    for (int kind = kTile256x128; kind < kGemmKinds; ++kind) {
        int64_t tiles = 0;
        for (int i = 0; i < count; ++i) tiles += tiles_of(kind, M[i], N[i]);
        if (tiles * 16 >= (1LL << 31)) continue;
        for (int64_t s = 1; s <= 16; ++s) {
            if (s > 1 && (kind == kTile64Waves || nk / s < 4 || tiles * s > 4 * kCus ||
                          tiles * s * gemm_kind_bm(kind) * gemm_kind_bn(kind) * 4 > room))
                break;
            const double t = cost_small(rates[kind], row, kind, tiles, nk, s, out_mb) * (kind == kTile128 ? list_128 : 1);
            if (t * margin < t_best) {
                t_best = t * margin;
                best.kind = kind;
                best.nsplit = (int)s;
            }
        }
    }
    if (time) *time = best.kind == kTile256 ? t_best : t_best / margin;
    return best;
}
// One product.  kRates take too little for what a split costs where the tiles are 64 x 64: they ask for twice the shares that are fastest, or for whole tiles
// of eight waves where shares are faster.  Where they end at such tiles and kOtherRates at shares, the latter's plan is taken.  Time of kRates' plan over that one, 600 such
// products of 128 - 8192 wide operands and 64 - 16384 rows, everything in the caches and weights from HBM: 64 x 64 in more shares 1.09, 1.12 (forward), 1.08, 1.11
// (input gradients) and 1.06, 1.09 (weight gradients), whole 64 x 64 tiles instead of shares 0.91, 1.26 (forward and input gradients).  M x N x K, weights from HBM, us:
// 605 x 384 x 2560 in 8 shares 12.9, in 4 11.2; 376 x 576 x 3328 9, 4 14.0, 11.8; weight gradient 576 x 512 x 2989 7, 3 14.6, 12.8; 191 x 320 x 1728 whole 11.4, in 6 9.0.
GemmPlan find_plan(Class cls, bool lines, int64_t M, int64_t N, int64_t nk, int64_t room) {
    const GemmPlan plan = find_plan(cls, lines, 1, &M, &N, nk, room);
    if (!lines || (plan.kind != kTile64 && plan.kind != kTile64Waves)) return plan;
    const GemmPlan other = find_plan(cls, false, 1, &M, &N, nk, room);
    return other.nsplit > 1 ? other : plan;
}
// A search takes 0.3 us and more, and each product of a step is asked for twice, when its workspace is sized and when it is launched: a thread remembers
// 256 products of a class by sizes and room, and 256 workspaces (below).  The planning of a layer's nine products, each sized and launched, 1167 tokens, h = 256,
// 768, 1024: 0.1 us each, the first time 4.4, 7.1, 6.3; with one slot for whatever room, where the two questions throw each other out, and the powers computed
// in every search 6.9, 10.8, 10.4 and 14, 21, 20.
uint64_t memo_slot(int64_t M, int64_t N, int64_t K, int64_t room) {
    return (uint64_t)(M * 0x9E3779B97F4A7C15ull ^ N * 0xC2B2AE3D27D4EB4Full ^ K * 0x165667B19E3779F9ull ^ room * 0xD6E8FEB86659FD93ull) >> 56;
}
thread_local int64_t searches = 0;  // (ezl_gemm_searches)
GemmPlan choose_plan(Class cls, int64_t M, int64_t N, int64_t K, int64_t room) {
    const int64_t nk = (K + BK - 1) / BK;
    struct Entry {
        int64_t M, N, K, room;
        GemmPlan plan;
    };
    static thread_local Entry memo[3][256] = {};
    Entry& e = memo[cls][memo_slot(M, N, K, room)];
    if (e.M != M || e.N != N || e.K != K || e.room != room) {
        e = {M, N, K, room, find_plan(cls, whole_lines(cls, M, N, K), M, N, nk, room)};
        ++searches;
    }
    return e.plan;
}
int64_t small_plan_bytes(const GemmPlan& p, int count, const int64_t* M, const int64_t* N) {
    int64_t tiles = 0;
    for (int i = 0; i < count; ++i) tiles += tiles_of(p.kind, M[i], N[i]);
    return p.nsplit > 1 ? tiles * p.nsplit * gemm_kind_bm(p.kind) * gemm_kind_bn(p.kind) * (int64_t)sizeof(float) : 0;
}
// Products that share a reduction length (q / k / v or gate / up of one input, and their weight gradients) in one launch?  Worth
// it where each of them leaves CUs idle: 1024 tokens at h = 256, q + k + v forward 3 x 4.7 us alone.  The launches of a long
// batch fill the chip one by one, with the better 256 x 256 tiles (at 4096 tokens and h = 4096 one launch for q / k / v
// measured 0.14 ms per four-layer step slower).  The estimates compare well; where each product alone takes 256 x 256 tiles they still
// flatter the one launch a little, which has to win by a twenty-fifth there.
// Estimated ratio -> measured time apart and together, us (T tokens, width / widths; f forward, w weight gradient):
//   smaller tiles alone     w 10604, 2176 / 2176, 2 x 512 0.76 -> 186, 132; f 1601, 4096 / 4096, 2 x 512 0.96 -> 85, 78; w 926, 6400 / 3 x 6400 0.98
//                           -> 314, 281; at worst f 15975, 1664 / 1664, 2 x 384 0.94 -> 121, 132
//   256 x 256, to 0.96      w 1910, 3072 / 3 x 3072 0.73 -> 170, 117; f 684, 4992 / 2 x 14744 0.92 -> 223, 199; w 4301, 4352 / 3 x 4352 0.95 -> 514,
//                           443; at worst f 12911, 640 / 2 x 2160 0.96 -> 80, 83
//   256 x 256, above        w 8316, 5888 / 5888, 2 x 1472 0.98 -> 868, 821; w 1221, 5504 / 3 x 5504 0.99 -> 255, 257; f 3298, 3840 / 2 x 11968 1.02
//                           -> 491, 531; f 5851, 1664 / 2 x 4512 1.05 -> 147, 178
// Over 240 groups of widths 256 - 8192 and 256 - 16384 tokens with estimated ratios of 0.7 - 1.1: 0.25 % (forward) and 0.39 % (weight gradients)
// behind the faster of the two on average; without the margin 0.31 and 0.33 %, with one of a tenth 0.79 and 0.88 %.
constexpr double kLaunchGap = 2.5;  // us between two launches of a stream: ramp down, ramp up
constexpr double kMargin256 = 0.96;
struct GroupTimes {
    GemmPlan plan;           // of the one launch
    double together, apart;  // estimated us
    bool one;
};
GroupTimes group_times(bool wgrad, int count, const int64_t* M, const int64_t* N, int64_t K, int64_t room, bool list_256 = false) {
    struct Entry {
        int64_t M[kMaxProblems], N[kMaxProblems], K, room;
        GroupTimes times;
        int count;
        bool wgrad, list_256;
    };
    static thread_local Entry memo[2][64] = {};  // (by list_256: group_bytes asks for one set of sizes both ways, each time)
    uint64_t hash = K * 0x165667B19E3779F9ull + 2 * count + wgrad;
    for (int i = 0; i < count; ++i) hash = (hash ^ (uint64_t)M[i]) * 0x9E3779B97F4A7C15ull + (uint64_t)N[i] * 0xC2B2AE3D27D4EB4Full;
    Entry& e = memo[list_256][hash >> 58];
    bool same = e.count == count && e.wgrad == wgrad && e.list_256 == list_256 && e.K == K && e.room == room;
    for (int i = 0; i < count && same; ++i) same = e.M[i] == M[i] && e.N[i] == N[i];
    if (!same) {
        const int64_t nk = (K + BK - 1) / BK;
        GroupTimes& g = e.times;
        g.apart = kLaunchGap * (count - 1);
        bool all_256 = true;
        for (int i = 0; i < count; ++i) {
            double t;
            all_256 = gemm_kind_large(find_plan(wgrad ? kWeightGradient : kForward, false, 1, &M[i], &N[i], nk, room, &t).kind) && all_256;
            g.apart += t;
            e.M[i] = M[i];
            e.N[i] = N[i];
        }
        g.plan = find_plan(wgrad ? kWeightGradient : kForward, false, count, M, N, nk, room, &g.together, list_256);
        if (all_256 && g.plan.kind != kTile256) g.together /= kMargin256;
        g.one = g.together < g.apart;
        e.K = K;
        e.room = room;
        e.count = count;
        e.wgrad = wgrad;
        e.list_256 = list_256;
    }
    return e.times;
}
bool group_plan(bool wgrad, int count, const int64_t* M, const int64_t* N, int64_t K, int64_t room, GemmPlan& plan, bool list_256 = false) {
    const GroupTimes g = group_times(wgrad, count, M, N, K, room, list_256);
    plan = g.plan;
    return g.one;
}
// workspace of a product's plan, whichever form it has; the 256 x 256 kernels' own where a launch has to fall back to them
int64_t find_bytes(int64_t M, int64_t N, int64_t K) {
    const int64_t nk = (K + BK - 1) / BK, tiles = tiles_of(kTile256, M, N);
    int64_t most = split_bytes(kTile256, false, tiles, nk);
    for (const Class cls : {kForward, kInputGradient, kWeightGradient}) {
        const bool lines = whole_lines(cls, M, N, K);
        if (cls == kInputGradient && !lines) continue;  // (the rates of a forward product)
        const GemmPlan q = find_plan(cls, lines, M, N, nk, INT64_MAX);
        ++searches;
        const int64_t large = split_bytes(kTile256, lines, tiles, nk);  // (also where its results have to be stored by the 8-wave kernel)
        most = large > most ? large : most;
        const int64_t small = gemm_kind_large(q.kind) ? split_bytes(q.kind, lines, tiles_of(q.kind, M, N), nk) : small_plan_bytes(q, 1, &M, &N);
        most = small > most ? small : most;
    }
    return most;
}
int64_t plan_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    struct Entry {
        int64_t M, N, K, bytes;
    };
    static thread_local Entry memo[256] = {};
    Entry& e = memo[memo_slot(M, N, K, 0)];
    if (e.M != M || e.N != N || e.K != K) e = {M, N, K, find_bytes(M, N, K)};
    return e.bytes;
}

// Which 256 x 256 kernel: the 4-wave one moves a third fewer LDS bytes and has its operands longer on the way; the 8-wave one hides more inside a
// tile, which shows where a launch is one round of short reductions.  Time of the 8-wave kernel over that of the 4-wave one, 17000 products of 256 - 96000 wide
// operands, by K tiles:
//                        2 - 7   8 - 15  16 - 31  32 - 63  64 - 127  128 - 399
//   forward, one round   1.01    1.03    1.04     1.09     1.15      1.19          several rounds 1.13 - 1.16
//   input gradient       0.99    0.98    0.98     1.00     1.04      1.06          1.06 - 1.15
//   ... over pairs       0.99    0.98    0.97     0.99     1.02      1.06          1.05 - 1.15
//   weight gradient      1.00    1.02    1.05     1.09     1.13      1.17          1.09 - 1.12
// (forward in one round under 48 K tiles: the 256 x 256 tiles are hardly ever the choice there; input gradients in one round of 64 - 127 K tiles: the 4 and 2 % are not
// taken, one line for both forms where both gain more).  The figures are of operands from HBM; with both in the caches one round of 8 - 47 K tiles of a weight gradient is 5 - 8 % slower on the
// 4-wave kernel, with one from HBM 3 - 7 % faster, with both 6 - 10 (90 products).  Several rounds of a weight gradient with the rows of B 16 KiB (or a
// multiple) apart, under 48 K tiles: 32000 x 8192 x 1536 0.94, 28672 x 8192 x 1536 0.96.
// items: workgroup-sized pieces of the launch; nk: K tiles of a piece; shares: pieces are shares of a reduction
enum class Form { forward, weight_gradient, input_gradient, input_gradient_segments };
bool w4_pays(Form form, int64_t nk, int64_t items, int64_t ldb, bool shares = false) {
    const bool rounds = items > kCus;
    switch (form) {
        case Form::forward: return nk >= 48 || rounds || (shares && nk >= 12);
        case Form::weight_gradient: return nk >= 48 || (nk >= 8 && !(rounds && ldb % 8192 == 0));
        default: return nk >= 128 || rounds || (shares && nk >= 12);
    }
}
// the same for a product's launch: one that is split tiles only is judged by the length of a share
bool w4_pays(Form form, const SplitPlan& plan, int64_t nk, int64_t ldb) {
    const bool shares = plan.nsplit > 1 && plan.full == 0;
    if (shares) nk /= plan.nsplit;
    return nk >= 2 && w4_pays(form, nk, plan.full + plan.rest * plan.nsplit, ldb, shares);
}
// Workgroups of a 4-wave launch: one per CU, each walking over its tiles (one per tile costs, by K tiles, 2 - 7 7 - 12 %, 8 - 31 3 - 8, 32 - 63 2 - 3, from 64 on 0 - 1).
dim3 w4_grid(int64_t items) { return dim3((unsigned)(items > kCus ? kCus : items)); }
// its stores: 16 bytes each, at 31-bit byte offsets inside a tile
template <typename OutT>
bool w4_stores_ok(const void* C, int64_t N, int64_t ldc) {
    const int vec = 16 / (int)sizeof(OutT);
    return N % vec == 0 && ldc % vec == 0 && ezl_aligned16(C) && ldc * (int64_t)sizeof(OutT) * BM < (1LL << 31);
}

// Lists of forward products or weight gradients on 256 x 256 tiles (4-wave kernel)
int64_t list_256_tiles(int count, const int64_t* M, const int64_t* N) {
    int64_t tiles = 0;
    for (int i = 0; i < count; ++i) tiles += tiles_of(kTile256, M[i], N[i]);
    return tiles;
}
bool list_256_pays(bool wgrad, int count, const int64_t* M, const int64_t* N, int64_t K) {
    const int64_t nk = (K + BK - 1) / BK, tiles = list_256_tiles(count, M, N);
    bool pays = tiles < (1LL << 26) && (nk >= 48 || (nk >= 16 && tiles > kCus));
    for (int i = 0; i < count; ++i) pays = pays && w4_pays(wgrad ? Form::weight_gradient : Form::forward, nk, tiles, N[i]);
    return pays;
}
int64_t list_256_bytes(int count, const int64_t* M, const int64_t* N, int64_t K) {
    const int64_t tiles = list_256_tiles(count, M, N);
    return split_bytes(kTile256, false, tiles, (K + BK - 1) / BK);
}
template <bool KC, typename OutT>
void launch_list_256(GemmSmallArgs& a, int count, void* workspace, int64_t workspace_bytes, hipStream_t st) {
    gemm_tile_grids({kTile256, 1}, a, count);
    const int nk = (a.K + BK - 1) / BK;
    const SplitPlan plan = make_plan(kTile256, false, a.ntiles, nk, workspace, workspace_bytes);
    const int items = plan.full + plan.rest * plan.nsplit;
#define EZL_LIST(KTAIL)                                                                                                                 \
    hipLaunchKernelGGL((gemm_w4_kernel<KC, KC, OutT, false, KTAIL, true>), w4_grid(items), dim3(256), 0, st, nullptr, nullptr,       \
                       (OutT*)nullptr, 0, 0, a.K, (int64_t)0, (int64_t)0, (int64_t)0, 0, 0, 0, items, plan, KSegments(), a)
    if (a.K % BK == 0) EZL_LIST(false);
    else EZL_LIST(true);
#undef EZL_LIST
    if (plan.nsplit > 1) {
        a.nsplit = plan.nsplit;
        a.partial = plan.partial;
        gemm_small_reduce(kTile256, sizeof(OutT) == 4, plan.full, a, st);
    }
}

// large tiles: the 4-wave kernel in either height, or the 8-wave one.  ktot: length of the whole reduction, from which the workspace was sized (the K tiles of
// several pairs can be one or two more)
template <bool A_KC, bool B_KC, typename OutT, bool MULTI, bool KTAIL>
void launch_large(int kind, bool lines, int64_t ktot, const void* A, const void* B, void* C, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int accumulate,
                  void* workspace, int64_t workspace_bytes, const KSegments& seg, hipStream_t st) {
    const int nk = MULTI ? seg.nk : (K + BK - 1) / BK;
    // (fp32 input gradients stay with the 8-wave kernel)
    constexpr bool HAS_W4 = A_KC ? B_KC || sizeof(OutT) == 2 : !B_KC;
    constexpr Form form = !A_KC ? Form::weight_gradient : (B_KC ? Form::forward : (MULTI ? Form::input_gradient_segments : Form::input_gradient));
    bool w4 = false;
    if constexpr (HAS_W4) w4 = w4_stores_ok<OutT>(C, N, ldc);
    constexpr bool HAS_192 = HAS_W4 && (!KTAIL || !A_KC || MULTI);  // (whole_lines: the others' reductions are whole K tiles)
    if (!w4 || !HAS_192) kind = kTile256;
    const int tiles_m = (int)((M + gemm_kind_bm(kind) - 1) / gemm_kind_bm(kind)), tiles_n = (N + BN - 1) / BN;
    const SplitPlan plan = make_plan(kind, lines, (int64_t)tiles_m * tiles_n, (ktot + BK - 1) / BK, workspace, workspace_bytes);
    const int items = plan.full + plan.rest * plan.nsplit;
    w4 = w4 && (kind == kTile192x256 || w4_pays(form, plan, nk, ldb));
    if constexpr (HAS_W4) {
#define EZL_W4(TBM)                                                                                                                            \
    hipLaunchKernelGGL((gemm_w4_kernel<A_KC, B_KC, OutT, MULTI, KTAIL, false, TBM>), w4_grid(items), dim3(256), 0, st, (const bf16_t*)A,     \
                       (const bf16_t*)B, (OutT*)C, M, N, K, lda, ldb, ldc, accumulate, tiles_m, tiles_n, items, plan, seg, NoList())
        if (w4 && kind == kTile192x256) {
            if constexpr (HAS_192) EZL_W4(192);
        } else if (w4) {
            EZL_W4(256);
        }
#undef EZL_W4
    }
    if (!w4)
        hipLaunchKernelGGL((gemm_d2l_kernel<A_KC, B_KC, OutT, MULTI, KTAIL>), dim3((unsigned)items), dim3(512), 0, st, (const bf16_t*)A,
                           (const bf16_t*)B, (OutT*)C, M, N, K, lda, ldb, ldc, accumulate, tiles_m, tiles_n, plan, seg);
#define EZL_REDUCE(TBM)                                                                                                                    \
    hipLaunchKernelGGL((gemm_split_reduce_kernel<OutT, TBM>), dim3((unsigned)(plan.rest * (TBM / kReduceRows))), dim3(256), 0, st, (OutT*)C, M, N, ldc, \
                       accumulate, tiles_m, tiles_n, plan)
    if (plan.nsplit > 1) {
        if (kind == kTile192x256) EZL_REDUCE(192);
        else EZL_REDUCE(256);
    }
#undef EZL_REDUCE
}
// the smaller-tile kernels store at 31-bit byte offsets inside a tile
template <typename OutT>
bool small_stores_ok(int64_t ldc) {
    return ldc * (int64_t)sizeof(OutT) * 256 < (1LL << 31);
}
template <bool A_KC, bool B_KC, typename OutT>
void launch(const void* A, const void* B, void* C, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int accumulate,
            void* workspace, int64_t workspace_bytes, hipStream_t st) {
    constexpr int form = A_KC ? (B_KC ? (sizeof(OutT) == 4 ? 4 : 0) : 1) : (sizeof(OutT) == 4 ? 2 : 3);
    constexpr Class cls = !A_KC ? kWeightGradient : (B_KC ? kForward : kInputGradient);
    const bool lines = whole_lines(cls, M, N, K);
    int kind = kTile256;
    if constexpr (A_KC ? B_KC || sizeof(OutT) == 2 : !B_KC) {
        if (small_stores_ok<OutT>(ldc)) {
            const GemmPlan plan = choose_plan(cls, M, N, K, workspace ? workspace_bytes : 0);
            kind = plan.kind;
            if (!gemm_kind_large(kind)) {
                GemmSmallArgs a = {};
                a.p[0] = {(const bf16_t*)A, (const bf16_t*)B, C, lda, ldb, ldc, M, N, 0, 0, 0, accumulate};
                a.K = K;
                a.partial = (float*)workspace;
                gemm_small_launch(form, false, plan, a, 1, st);
                return;
            }
        }
    }
    if (K % BK == 0)
        launch_large<A_KC, B_KC, OutT, false, false>(kind, lines, K, A, B, C, M, N, K, lda, ldb, ldc, accumulate, workspace, workspace_bytes, KSegments(), st);
    else
        launch_large<A_KC, B_KC, OutT, false, true>(kind, lines, K, A, B, C, M, N, K, lda, ldb, ldc, accumulate, workspace, workspace_bytes, KSegments(), st);
}

// C = 0 for an empty reduction (a fill kernel rather than a memset node, so the call can be captured into a graph)
template <typename OutT>
__global__ __launch_bounds__(256) void zero_c_kernel(OutT* __restrict__ C, int64_t M, int64_t N, int64_t ldc) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < M * N; i += (int64_t)gridDim.x * 256)
        C[(i / N) * ldc + (i % N)] = (OutT)0.0f;
}

}  // namespace


static int check_operands(const void* A, const void* B, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int a_kc,
                          int b_kc) {
    EZL_REQUIRE(A && B, EZL_EINVAL, "ezl_gemm_bf16: null pointer");
    EZL_REQUIRE(ezl_aligned16(A) && ezl_aligned16(B) && lda % 8 == 0 && ldb % 8 == 0, EZL_EINVAL,
                "ezl_gemm_bf16: operands must be 16-byte aligned with leading dimensions that are multiples of 8");
    // every 128-bit chunk must lie wholly inside or wholly outside the matrix
    EZL_REQUIRE(a_kc ? (K % 8 == 0) : (M % 8 == 0), EZL_EUNSUPPORTED, "ezl_gemm_bf16: contiguous extent of A must be a multiple of 8");
    EZL_REQUIRE(b_kc ? (K % 8 == 0) : (N % 8 == 0), EZL_EUNSUPPORTED, "ezl_gemm_bf16: contiguous extent of B must be a multiple of 8");
    EZL_REQUIRE(lda >= (a_kc ? K : M) && ldb >= (b_kc ? K : N) && ldc >= N, EZL_EINVAL, "ezl_gemm_bf16: leading dimension too small");
    // 32-bit byte offsets inside one 256-row (or 64-k-row) tile; the tile bases advance in 64 bits
    EZL_REQUIRE(lda < (1LL << 22) && ldb < (1LL << 22) && M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31), EZL_EUNSUPPORTED,
                "ezl_gemm_bf16: a dimension of 2^31 or more, or a leading dimension of 2^22 or more");
    const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    EZL_REQUIRE(tiles < (1LL << 31), EZL_EUNSUPPORTED, "ezl_gemm_bf16: too many tiles");
    return EZL_OK;
}

// a_kc / b_kc: 1 if the operand's reduction index is its contiguous one
//   A: a_kc ? A[m * lda + k] : A[k * lda + m]        B: b_kc ? B[n * ldb + k] : B[k * ldb + n]
// out_dtype: 0 bf16, 1 fp32, 2 fp32 holding bf16 values (forward form, no accumulation).  accumulate: C += A*B instead of C = A*B.
// bytes of workspace with which a launch of this shape evens out a mostly empty last round of tiles (0: none needed)
extern "C" int64_t ezl_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) { return plan_bytes(M, N, K); }

extern "C" int ezl_gemm_bf16(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                             int64_t ldc, int a_kc, int b_kc, int out_dtype, int accumulate, void* workspace,
                             int64_t workspace_bytes, void* stream) {
    EZL_REQUIRE(M >= 0 && N >= 0 && K >= 0, EZL_EINVAL, "ezl_gemm_bf16: negative size");
    EZL_REQUIRE(out_dtype == 0 || out_dtype == 1 || (out_dtype == 2 && a_kc && b_kc && !accumulate), EZL_EUNSUPPORTED,
                "ezl_gemm_bf16: out_dtype must be 0 (bf16), 1 (fp32) or, for an overwriting forward product, 2 (bf16 values as fp32)");
    if (accumulate) accumulate = 1;
    if (out_dtype == 2) {
        out_dtype = 1;
        accumulate = kRoundResult;
    }
    if (M == 0 || N == 0) return EZL_OK;
    EZL_REQUIRE(C, EZL_EINVAL, "ezl_gemm_bf16: null pointer");
    if (K == 0) {  // empty reduction (a weight gradient over zero tokens): C = 0, or C unchanged when accumulating
        EZL_REQUIRE(ldc >= N, EZL_EINVAL, "ezl_gemm_bf16: leading dimension too small");
        if (accumulate != 1) {
            if (out_dtype == 0) hipLaunchKernelGGL(zero_c_kernel<bf16_t>, dim3(256), dim3(256), 0, (hipStream_t)stream, (bf16_t*)C, M, N, ldc);
            else hipLaunchKernelGGL(zero_c_kernel<float>, dim3(256), dim3(256), 0, (hipStream_t)stream, (float*)C, M, N, ldc);
            EZL_LAUNCH_CHECK("ezl_gemm_bf16(zero)");
        }
        return EZL_OK;
    }
    if (const int rc = check_operands(A, B, M, N, K, lda, ldb, ldc, a_kc, b_kc)) return rc;
    hipStream_t st = (hipStream_t)stream;
    EZL_REQUIRE(!workspace || ezl_aligned16(workspace), EZL_EINVAL, "ezl_gemm_bf16: workspace must be 16-byte aligned");
#define EZL_GEMM_CASE(AK, BKC, OT) \
    launch<AK, BKC, OT>(A, B, C, (int)M, (int)N, (int)K, lda, ldb, ldc, accumulate, workspace, workspace_bytes, st)
    if (out_dtype == 0) {
        if (a_kc && b_kc) EZL_GEMM_CASE(true, true, bf16_t);
        else if (a_kc && !b_kc) EZL_GEMM_CASE(true, false, bf16_t);
        else if (!a_kc && !b_kc) EZL_GEMM_CASE(false, false, bf16_t);
        else EZL_GEMM_CASE(false, true, bf16_t);
    } else {
        if (a_kc && b_kc) EZL_GEMM_CASE(true, true, float);
        else if (a_kc && !b_kc) EZL_GEMM_CASE(true, false, float);
        else if (!a_kc && !b_kc) EZL_GEMM_CASE(false, false, float);
        else EZL_GEMM_CASE(false, true, float);
    }
#undef EZL_GEMM_CASE
    EZL_LAUNCH_CHECK("ezl_gemm_bf16");
    return EZL_OK;
}

int gemm_forward_add(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, void* workspace, int64_t workspace_bytes, void* stream) {
    EZL_REQUIRE(M > 0 && N > 0 && K > 0 && C, EZL_EINVAL, "ezl_gemm_bf16: null pointer or empty product");
    if (const int rc = check_operands(A, B, M, N, K, K, K, N, 1, 1)) return rc;
    EZL_REQUIRE(!workspace || ezl_aligned16(workspace), EZL_EINVAL, "ezl_gemm_bf16: workspace must be 16-byte aligned");
    launch<true, true, bf16_t>(A, B, C, (int)M, (int)N, (int)K, K, K, N, 1 | kRoundResult, workspace, workspace_bytes, (hipStream_t)stream);
    EZL_LAUNCH_CHECK("ezl_gemm_bf16");
    return EZL_OK;
}

// C (=|+=) sum_i A[i] * B[i] over `count` operand pairs that share M, N and the leading dimensions; K[i] is the reduction
// length of pair i.  The input gradient dx = sum_i dy_i W_i of linears that share their input is one such sum.  With up to
// three pairs in the (a_kc = 1, b_kc = 0, bf16 output) form and every K[i] positive it is a single launch that adds the
// products in fp32 and rounds once; otherwise the pairs go out as ezl_gemm_bf16 calls that accumulate into C.
extern "C" int ezl_gemm_bf16_ksplit(int count, const void* const* A, const void* const* B, void* C, int64_t M, int64_t N,
                                    const int64_t* K, int64_t lda, int64_t ldb, int64_t ldc, int a_kc, int b_kc, int out_dtype,
                                    int accumulate, void* workspace, int64_t workspace_bytes, void* stream) {
    EZL_REQUIRE(count >= 1 && A && B && K, EZL_EINVAL, "ezl_gemm_bf16_ksplit: bad count or null argument array");
    accumulate = accumulate ? 1 : 0;  // (the kernels take a bit field)
    bool one_launch = count <= 3 && a_kc == 1 && b_kc == 0 && out_dtype == 0 && M > 0 && N > 0, tail = false;
    int64_t ktot = 0;
    for (int i = 0; i < count; ++i) {
        EZL_REQUIRE(K[i] >= 0, EZL_EINVAL, "ezl_gemm_bf16_ksplit: negative size");
        one_launch = one_launch && K[i] > 0;
        tail = tail || K[i] % BK != 0;
        ktot += K[i];
    }
    if (!one_launch || count == 1) {
        for (int i = 0; i < count; ++i)
            if (const int rc = ezl_gemm_bf16(A[i], B[i], C, M, N, K[i], lda, ldb, ldc, a_kc, b_kc, out_dtype, i == 0 ? accumulate : 1,
                                             workspace, workspace_bytes, stream))
                return rc;
        return EZL_OK;
    }
    EZL_REQUIRE(C, EZL_EINVAL, "ezl_gemm_bf16: null pointer");
    for (int i = 0; i < count; ++i) {
        EZL_REQUIRE(A[i] && B[i], EZL_EINVAL, "ezl_gemm_bf16: null pointer");
        EZL_REQUIRE(ezl_aligned16(A[i]) && ezl_aligned16(B[i]) && lda % 8 == 0 && ldb % 8 == 0, EZL_EINVAL,
                    "ezl_gemm_bf16: operands must be 16-byte aligned with leading dimensions that are multiples of 8");
        EZL_REQUIRE(K[i] % 8 == 0, EZL_EUNSUPPORTED, "ezl_gemm_bf16: contiguous extent of A must be a multiple of 8");
        EZL_REQUIRE(lda >= K[i] && lda < (1LL << 22) && ldb < (1LL << 22), EZL_EUNSUPPORTED,
                    "ezl_gemm_bf16: leading dimension too small, or 2^22 or more");
    }
    EZL_REQUIRE(N % 8 == 0 && ldb >= N && ldc >= N && M < (1LL << 31) && N < (1LL << 31) && ktot < (1LL << 31), EZL_EUNSUPPORTED,
                "ezl_gemm_bf16: contiguous extent of B must be a multiple of 8");
    const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    EZL_REQUIRE(tiles < (1LL << 31), EZL_EUNSUPPORTED, "ezl_gemm_bf16: too many tiles");
    KSegments seg;
    auto ktiles = [&](int i) { return (int)((K[i] + BK - 1) / BK); };
    seg.A1 = (const bf16_t*)A[1]; seg.B1 = (const bf16_t*)B[1]; seg.K1 = (int)K[1];
    seg.t1 = ktiles(0);
    seg.t2 = seg.nk = seg.t1 + ktiles(1);
    if (count > 2) seg.nk += ktiles(2);
    seg.A2 = count > 2 ? (const bf16_t*)A[2] : seg.A1; seg.B2 = count > 2 ? (const bf16_t*)B[2] : seg.B1; seg.K2 = count > 2 ? (int)K[2] : 0;
    EZL_REQUIRE(!workspace || ezl_aligned16(workspace), EZL_EINVAL, "ezl_gemm_bf16: workspace must be 16-byte aligned");
    int kind = kTile256;
    if (small_stores_ok<bf16_t>(ldc)) {
        const GemmPlan small = choose_plan(kInputGradient, M, N, ktot, workspace ? workspace_bytes : 0);
        kind = small.kind;
        if (!gemm_kind_large(kind)) {
            GemmSmallArgs a = {};
            a.p[0] = {(const bf16_t*)A[0], (const bf16_t*)B[0], C, lda, ldb, ldc, (int)M, (int)N, 0, 0, 0, accumulate};
            a.K = (int)K[0];
            a.partial = (float*)workspace;
            a.seg = seg;
            gemm_small_launch(1, true, small, a, 1, (hipStream_t)stream);
            EZL_LAUNCH_CHECK("ezl_gemm_bf16_ksplit");
            return EZL_OK;
        }
    }
    (tail ? launch_large<true, false, bf16_t, true, true> : launch_large<true, false, bf16_t, true, false>)(
        kind, whole_lines(kInputGradient, M, N, ktot), ktot, A[0], B[0], C, (int)M, (int)N, (int)K[0], lda, ldb, ldc, accumulate, workspace, workspace_bytes, seg, (hipStream_t)stream);
    EZL_LAUNCH_CHECK("ezl_gemm_bf16_ksplit");
    return EZL_OK;
}

namespace {
// Whether two results of a group share memory (one weight used by two projections: one gradient buffer): in one launch their tiles
// would be read and written in any order.  Address ranges are compared, so interleaved column blocks count as sharing.
bool results_meet(int count, void* const* C, const int64_t* M, const int64_t* N, const int64_t* ldc, int64_t size) {
    for (int i = 1; i < count; ++i)
        for (int j = 0; j < i; ++j) {
            const char *a = (const char*)C[i], *b = (const char*)C[j];
            if (a < b + ((M[j] - 1) * ldc[j] + N[j]) * size && b < a + ((M[i] - 1) * ldc[i] + N[i]) * size) return true;
        }
    return false;
}
}  // namespace

// Up to three independent products C[i] (=|+=) A[i] * B[i] over one reduction length K in one launch; one after the other where their
// results share memory or have rows too far apart.
// ezl_gemm_group_form_workspace_bytes: -1 where separate ezl_gemm_bf16 calls are estimated to be faster, else the workspace.
constexpr int kGroupMax = 3;  // q / k / v
static_assert(kGemmListMax == kMaxProblems, "a list goes out in one launch");
extern "C" int64_t ezl_gemm_group_form_workspace_bytes(int a_kc, int count, const int64_t* M, const int64_t* N, int64_t K) {
    if (count < 2 || count > kGroupMax || !M || !N || K <= 0) return -1;
    for (int i = 0; i < count; ++i)
        if (M[i] <= 0 || N[i] <= 0 || M[i] >= (1LL << 31) || N[i] >= (1LL << 31)) return -1;
    GemmPlan plan;
    bool one = group_plan(!a_kc, count, M, N, K, INT64_MAX, plan);
    int64_t bytes = small_plan_bytes(plan, count, M, N);  // (an input gradient, or results that the large tiles cannot store)
    if (a_kc && list_256_pays(false, count, M, N, K)) {
        one = group_plan(false, count, M, N, K, INT64_MAX, plan, true);
        const int64_t large = plan.kind == kTile256 ? list_256_bytes(count, M, N, K) : 0;
        bytes = bytes > large ? bytes : large;
    }
    return one ? bytes : -1;
}
// The form is not said: products with K = N are taken for the forward of square weights, others for weight gradients (gate and up are
// long in both).  The workspace is enough for either form's plan.
extern "C" int64_t ezl_gemm_group_workspace_bytes(int count, const int64_t* M, const int64_t* N, int64_t K) {
    const int64_t fwd = ezl_gemm_group_form_workspace_bytes(1, count, M, N, K), wgrad = ezl_gemm_group_form_workspace_bytes(0, count, M, N, K);
    if (fwd < 0 && wgrad < 0) return -1;
    if ((N[0] == K ? fwd : wgrad) < 0) return -1;
    return fwd > wgrad ? fwd : wgrad;
}

extern "C" int ezl_gemm_bf16_group(int count, const void* const* A, const void* const* B, void* const* C, const int64_t* M, const int64_t* N,
                                   int64_t K, const int64_t* lda, const int64_t* ldb, const int64_t* ldc, int a_kc, int b_kc, int out_dtype,
                                   const int* accumulate, void* workspace, int64_t workspace_bytes, void* stream) {
    EZL_REQUIRE(count <= kGroupMax, EZL_EINVAL, "ezl_gemm_bf16_group: bad count, null argument array or empty reduction");
    return gemm_list(count, A, B, C, M, N, K, lda, ldb, ldc, a_kc, b_kc, out_dtype, accumulate, workspace, workspace_bytes, stream);
}

// A decoder layer's weight gradients all reduce over its tokens.  Behind one another each of them is a launch that fills a part of the
// chip (2 x 512 tokens at h = 256: 16 to 132 workgroups, four launches of 8 us), as one list of tiles they fill it together.
int64_t gemm_list_workspace_bytes(int pieces, const int* counts, const int64_t* M, const int64_t* N, int64_t K, bool beyond_cache) {
    double in_pieces = kLaunchGap * (pieces - 1);
    int count = 0;
    for (int p = 0; p < pieces; ++p) {
        const GroupTimes g = group_times(true, counts[p], M + count, N + count, K, INT64_MAX);
        in_pieces += g.one ? g.together : g.apart;
        count += counts[p];
    }
    const GroupTimes all = group_times(true, count, M, N, K, INT64_MAX, list_256_pays(true, count, M, N, K));
    if (all.together >= in_pieces || (beyond_cache && all.plan.kind != kTile256)) return -1;
    return all.plan.kind == kTile256 ? list_256_bytes(count, M, N, K) : small_plan_bytes(all.plan, count, M, N);
}

int gemm_list(int count, const void* const* A, const void* const* B, void* const* C, const int64_t* M, const int64_t* N, int64_t K,
              const int64_t* lda, const int64_t* ldb, const int64_t* ldc, int a_kc, int b_kc, int out_dtype, const int* accumulate,
              void* workspace, int64_t workspace_bytes, void* stream) {
    EZL_REQUIRE(count >= 1 && count <= kMaxProblems && A && B && C && M && N && lda && ldb && ldc && accumulate && K > 0, EZL_EINVAL,
                "ezl_gemm_bf16_group: bad count, null argument array or empty reduction");
    EZL_REQUIRE((out_dtype == 0 && (a_kc || !b_kc)) || (out_dtype == 1 && !a_kc && !b_kc), EZL_EUNSUPPORTED,
                "ezl_gemm_bf16_group: forms are forward, input gradient and weight gradient");
    EZL_REQUIRE(!workspace || ezl_aligned16(workspace), EZL_EINVAL, "ezl_gemm_bf16_group: workspace must be 16-byte aligned");
    GemmSmallArgs a = {};
    int64_t tiles = 0;
    bool apart = false;
    for (int i = 0; i < count; ++i) {
        EZL_REQUIRE(C[i] && M[i] > 0 && N[i] > 0, EZL_EINVAL, "ezl_gemm_bf16_group: null pointer or empty product");
        if (const int rc = check_operands(A[i], B[i], M[i], N[i], K, lda[i], ldb[i], ldc[i], a_kc, b_kc)) return rc;
        // (rows of C too far apart for the smaller tiles' stores: ezl_gemm_bf16 has kernels for them)
        apart = apart || !(out_dtype == 0 ? small_stores_ok<bf16_t>(ldc[i]) : small_stores_ok<float>(ldc[i]));
        a.p[i] = {(const bf16_t*)A[i], (const bf16_t*)B[i], C[i], lda[i], ldb[i], ldc[i], (int)M[i], (int)N[i], 0, 0, 0, accumulate[i] ? 1 : 0};
        tiles += tiles_of(kTile64, M[i], N[i]);
    }
    EZL_REQUIRE(tiles < (1LL << 27), EZL_EUNSUPPORTED, "ezl_gemm_bf16_group: too many tiles");
    if (apart || results_meet(count, C, M, N, ldc, out_dtype == 0 ? 2 : 4)) {
        for (int i = 0; i < count; ++i)
            if (const int rc = ezl_gemm_bf16(A[i], B[i], C[i], M[i], N[i], K, lda[i], ldb[i], ldc[i], a_kc, b_kc, out_dtype, accumulate[i],
                                             workspace, workspace_bytes, stream))
                return rc;
        return EZL_OK;
    }
    GemmPlan plan;
    bool list_256 = (a_kc ? b_kc && count > 1 : count > kGroupMax) && list_256_pays(!a_kc, count, M, N, K);
    for (int i = 0; i < count; ++i) list_256 = list_256 && (out_dtype ? w4_stores_ok<float> : w4_stores_ok<bf16_t>)(C[i], N[i], ldc[i]);
    group_plan(!a_kc, count, M, N, K, INT64_MAX, plan, list_256);
    a.K = (int)K;
    if (list_256 && plan.kind == kTile256) {
        (a_kc ? launch_list_256<true, bf16_t> : (out_dtype ? launch_list_256<false, float> : launch_list_256<false, bf16_t>))(
            a, count, workspace, workspace_bytes, (hipStream_t)stream);
        EZL_LAUNCH_CHECK("ezl_gemm_bf16_group");
        return EZL_OK;
    }
    if (small_plan_bytes(plan, count, M, N) > (workspace ? workspace_bytes : 0)) group_plan(!a_kc, count, M, N, K, 0, plan);
    if (gemm_kind_large(plan.kind)) plan = {kTile256x128, 1};  // (a group of one: these kernels take one or more)
    a.partial = (float*)workspace;
    const int form = a_kc ? (b_kc ? 0 : 1) : (out_dtype == 1 ? 2 : 3);
    gemm_small_launch(form, false, plan, a, count, (hipStream_t)stream);
    EZL_LAUNCH_CHECK("ezl_gemm_bf16_group");
    return EZL_OK;
}

extern "C" int64_t ezl_gemm_searches(void) { return searches; }
extern "C" int ezl_gemm_plan(int form, int count, const int64_t* M, const int64_t* N, int64_t K, int* rows, int* cols, int* split, int* waves) {
    if (form < 0 || form > 3 || count < 1 || count > kMaxProblems || (form > 1 && count > 1) || !M || !N || K <= 0 || !rows || !cols || !split || !waves)
        return -1;
    for (int i = 0; i < count; ++i)
        if (M[i] <= 0 || N[i] <= 0 || M[i] >= (1LL << 31) || N[i] >= (1LL << 31)) return -1;
    const bool wgrad = form == 1;
    const Class cls = wgrad ? kWeightGradient : (form == 0 ? kForward : kInputGradient);
    const Form forms[4] = {Form::forward, Form::weight_gradient, Form::input_gradient, Form::input_gradient_segments};
    const int64_t nk = (K + BK - 1) / BK;
    GemmPlan plan;
    bool one = true;
    if (count == 1) {
        plan = choose_plan(cls, M[0], N[0], K, INT64_MAX);
    } else {
        one = group_plan(wgrad, count, M, N, K, INT64_MAX, plan, (!wgrad || count > kGroupMax) && list_256_pays(wgrad, count, M, N, K));
    }
    *rows = kKindRows[plan.kind];
    *cols = kKindCols[plan.kind];
    *split = plan.nsplit;
    *waves = plan.kind == kTile64Waves ? 8 : 4;
    if (gemm_kind_large(plan.kind)) {
        const int64_t tiles = count == 1 ? tiles_of(plan.kind, M[0], N[0]) : list_256_tiles(count, M, N);
        const SplitPlan p = make_plan(plan.kind, count == 1 && whole_lines(cls, M[0], N[0], K), tiles, nk, (void*)16, INT64_MAX);
        *split = p.nsplit;
        if (count == 1 && plan.kind == kTile256) *waves = w4_pays(forms[form], p, nk, form == 0 ? K : N[0]) ? 4 : 8;
    }
    return one;
}
