// GEMM kernels with smaller tiles than gemm.hip's 256 x 256, for products that do not fill the chip with those: short batches,
// narrow layers, weight gradients of narrow layers.  Same operand forms, LDS layouts and fragments.
//
// What a tile shape costs: the CU's address unit takes 16 cycles per 1 KiB wave load, so a 64-wide K tile of the operands
// takes 16 (BM + BN) / 8 cycles to fetch and BM BN / 32 cycles of MFMA (16x16x32, 16 cycles each, four SIMDs).  256 x 256:
// 1024 against 2048; 256 x 128: 768 against 1024; 128 x 128: 512 against 512; 64 x 64: 256 against 128.
// The smaller the tile, the more the fetch binds; what it buys is workgroups.
#include "gemm_tile.h"

namespace {

template <int N>
__device__ __forceinline__ void wait_loads() {  // all but the N newest loads of this wave have landed
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
// A stage's place in LDS, made opaque: the fragment reads go through restrict-qualified pointers, so without it the compiler may
// take a re-read of the same address for the value it read before the stage was refilled.
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+s"(x));
    return x;
}
// workgroup id -> (tile, part): XCD-aware, parts outermost, so that an XCD's workgroups share operand bands and K range
__device__ __forceinline__ void tile_and_part(const GemmSmallArgs& a, int& tile, int& part) {
    const int total = a.ntiles * a.nsplit;
    const int per = total >> 3, rem = total & 7, xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    tile = xcd * per + (xcd < rem ? xcd : rem) + idx;
    part = tile / a.ntiles;
    tile -= part * a.ntiles;
}
__device__ __forceinline__ GemmProblem problem_of(const GemmSmallArgs& a, int tile) {
    int i = 0;
#pragma unroll
    for (int j = 1; j < kMaxProblems; ++j) i += tile >= a.first[j];
    return a.p[i];
}

template <typename OutT>
__device__ __forceinline__ bool vector_stores(const GemmProblem& p) {
    return p.N % 8 == 0 && p.ldc % (16 / (int)sizeof(OutT)) == 0 && ((uintptr_t)p.C & 15) == 0;
}
template <bool FORWARD, int TM, int TN, typename OutT>
__device__ __forceinline__ void store_tile(const f32x4 (&acc)[TM][TN], const GemmProblem& p, int m0, int n0, int row0, int col0, int lane) {
    OutT* C = (OutT*)p.C + (int64_t)m0 * p.ldc + n0;
    const int mrem = p.M - m0 < 256 ? p.M - m0 : 256, nrem = p.N - n0;  // (no tile is taller: the range fits 31 bits)
    if (vector_stores<OutT>(p)) store_tile_flags<TM, TN, OutT, true, FORWARD>(acc, C, p.ldc, mrem, nrem, row0, col0, lane, p.accumulate);
    else store_tile_flags<TM, TN, OutT, false, FORWARD>(acc, C, p.ldc, mrem, nrem, row0, col0, lane, p.accumulate);
}

// this workgroup's share of the reduction, as a dense fp32 tile; small_reduce_kernel adds the shares
template <int TM, int TN, int TBM, int TBN>
__device__ __forceinline__ void store_partial(const f32x4 (&acc)[TM][TN], const GemmSmallArgs& a, int tile, int part, int row0, int col0, int lane) {
    float* t = a.partial + ((size_t)tile * a.nsplit + part) * (size_t)(TBM * TBN);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            *reinterpret_cast<f32x4*>(t + (row0 + i * 16 + (lane & 15)) * TBN + col0 + j * 16 + 4 * (lane >> 4)) = acc[i][j];
}

// this workgroup's K tiles of nk in all: kt0 .. kt0 + (returned count) - 1
__device__ __forceinline__ int share_of(int nk, int part, int nsplit, int& kt0) {
    kt0 = (int)((int64_t)nk * part / nsplit);
    return (int)((int64_t)nk * (part + 1) / nsplit) - kt0;
}

template <int TM, int TN>
__device__ __forceinline__ void zero_acc(f32x4 (&acc)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
}

// =================================================================================================
// 256 x 128 and 192 x 128 tiles, 2 x 2 waves, three LDS stages
// =================================================================================================
// The 4-wave kernel of gemm.hip (one wave per SIMD, one MFMA per compile-time step) with smaller tiles.  The three stages (256 x 128:
// 144 KiB) let the wave loads of a K tile (12) go out over both phases, one every fifth MFMA (the address unit needs 48 of the
// 64 MFMA slots of a K tile), two K tiles ahead of their use; a stage is free from the barrier in front of its K tile's second
// phase on, because that phase works on fragments already in registers.
template <bool A_KC, bool B_KC, typename OutT, bool MULTI, bool KTAIL, int TBM, int TBN>
__global__ __launch_bounds__(256, 1) void gemm_wide_kernel(const GemmSmallArgs args) {
    constexpr int TM = TBM / 32, TN = TBN / 32;
    constexpr int STAGE = (TBM + TBN) * BK;
    __shared__ __attribute__((aligned(1024))) bf16_t smem[3 * STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tile, part;
    tile_and_part(args, tile, part);
    const GemmProblem p = problem_of(args, tile);
    int tm, tn;
    tile_of(tile - p.first, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * TBM, n0 = tn * TBN;
    const int arow = (wave >> 1) * (TBM / 2), brow = (wave & 1) * (TBN / 2);
    TileLoader<A_KC, TBM, 4, KTAIL> la;
    TileLoader<B_KC, TBN, 4, KTAIL> lb;
    const int64_t a_blk = A_KC ? (int64_t)m0 * p.lda : (int64_t)m0;
    const int64_t b_blk = B_KC ? (int64_t)n0 * p.ldb : (int64_t)n0;
    la.init(lane, wave, p.M - m0, p.lda);
    lb.init(lane, wave, p.N - n0, p.ldb);
    const int64_t astep = A_KC ? BK : (int64_t)BK * p.lda;
    const int64_t bstep = B_KC ? BK : (int64_t)BK * p.ldb;
    int kt0;
    const int nk = share_of(MULTI ? args.seg.nk : (args.K + BK - 1) / BK, part, args.nsplit, kt0);
    f32x4 acc[TM][TN];
    zero_acc(acc);

    constexpr int NA = TM, NL = TM + TN;  // wave loads per K tile: A, and A + B
    constexpr int NF = TM + TN;          // fragments per k half
    constexpr int NM = TM * TN;          // MFMAs per phase
    constexpr int RSTEP = 2, LSTEP = 2 * NM / NL;  // a fragment read every RSTEP MFMAs of a phase, a load every LSTEP of both
    static_assert(RSTEP * NF <= NM + RSTEP - 1, "all fragments of a k half are read during the other one");
    bf16x8 fa[2][TM], fb[2][TN];
    auto read_frag = [&](const bf16_t* sA, int ks, int buf, auto F) {
        constexpr int f = decltype(F)::value;
        if constexpr (f < TN) fb[buf][f] = sfrag<B_KC, TBN>(sA + TBM * BK, brow + f * 16, ks, lane);
        else fa[buf][f - TN] = sfrag<A_KC, TBM>(sA, arow + (f - TN) * 16, ks, lane);
    };
    __amdgpu_buffer_rsrc_t ga, gb;
    int kv = BK;
    auto tile_bases = [&](int t) {
        const bf16_t *Ab, *Bb;
        t += kt0;
        pick_segment<MULTI>(p.A, p.B, args.K, args.seg, t, kv, Ab, Bb);
        ga = la.base(Ab + a_blk + (int64_t)t * astep);
        gb = lb.base(Bb + b_blk + (int64_t)t * bstep);
    };
    auto issue_load = [&](bf16_t* st, auto L) {
        constexpr int l = decltype(L)::value;
        if constexpr (l < NA) la.template issue_at<l>(ga, st, lane, wave, kv);
        else lb.template issue_at<l - NA>(gb, st + TBM * BK, lane, wave, kv);
    };
    auto issue_tile = [&](int t, bf16_t* st) {
        tile_bases(t);
        static_for<0, NL>([&](auto L) { issue_load(st, L); });
    };
    int s0 = 0, s1 = STAGE, s2 = 2 * STAGE;  // stages of K tiles kt, kt + 1, kt + 2
    issue_tile(0, smem + s0);
    if (nk > 1) issue_tile(1, smem + s1);
    if (nk > 2) issue_tile(2, smem + s2);
    if (nk > 2) wait_loads<2 * NL>();
    else wait_loads<0>();
    wave_barrier();
    static_for<0, NF>([&](auto F) { read_frag(smem + s0, 0, 0, F); });

    typedef std::true_type yes;
    typedef std::false_type no;
    // k half 1 of a K tile (stage sA) is read while half 0 is multiplied, half 0 of the next one (sN) while half 1 is
    auto phase_a = [&](const bf16_t* sA, bf16_t* sL, auto DO_LOAD) {
        static_for<0, NM>([&](auto S) {
            constexpr int m = decltype(S)::value, i = m / TN, j = m % TN, g = NM + m;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[0][j], fa[0][i], acc[i][j], 0, 0, 0);
            if constexpr (m % RSTEP == 0 && m / RSTEP < NF) read_frag(sA, 1, 1, std::integral_constant<int, m / RSTEP>{});
            if constexpr (decltype(DO_LOAD)::value && g % LSTEP == LSTEP - 1 && g / LSTEP < NL) issue_load(sL, std::integral_constant<int, g / LSTEP>{});
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto phase_b = [&](const bf16_t* sN, bf16_t* sL, auto HAS_NEXT, auto DO_LOAD) {
        static_for<0, NM>([&](auto S) {
            constexpr int m = decltype(S)::value, i = m / TN, j = m % TN;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[1][j], fa[1][i], acc[i][j], 0, 0, 0);
            if constexpr (decltype(HAS_NEXT)::value && m % RSTEP == 0 && m / RSTEP < NF) read_frag(sN, 0, 0, std::integral_constant<int, m / RSTEP>{});
            if constexpr (decltype(DO_LOAD)::value && m % LSTEP == LSTEP - 1 && m / LSTEP < NL) issue_load(sL, std::integral_constant<int, m / LSTEP>{});
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto publish = [&](auto LEFT) {  // this wave's fragment reads are done and all but its LEFT newest loads have landed
        constexpr int left = decltype(LEFT)::value;
        __builtin_amdgcn_s_waitcnt(0x0070 | (left & 15) | ((left >> 4) << 14));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto rotate = [&]() {
        const int x = s0;
        s0 = s1; s1 = s2; s2 = opaque(x);
    };
    phase_a(smem + s0, smem, no{});
    if (nk > 2) publish(std::integral_constant<int, NL>{});
    else publish(std::integral_constant<int, 0>{});
    int kt = 0;
    for (; kt + 3 < nk; ++kt) {
        tile_bases(kt + 3);
        phase_b(smem + s1, smem + s0, yes{}, yes{});
        phase_a(smem + s1, smem + s0, yes{});
        publish(std::integral_constant<int, NL>{});
        rotate();
    }
    for (; kt + 1 < nk; ++kt) {
        phase_b(smem + s1, smem, yes{}, no{});
        phase_a(smem + s1, smem, no{});
        publish(std::integral_constant<int, 0>{});
        rotate();
    }
    phase_b(smem, smem, no{}, no{});
    if (args.nsplit > 1) store_partial<TM, TN, TBM, TBN>(acc, args, tile, part, arow, brow, lane);
    else store_tile<A_KC && B_KC, TM, TN, OutT>(acc, p, m0, n0, arow, brow, lane);
}

// =================================================================================================
// square tiles of 128 or 64, 2 x 2 waves, ST LDS stages, more than one workgroup per CU
// =================================================================================================
// One barrier per K tile and no hand-laid schedule: the CU's other workgroups cover a wave's waits.  128: two stages (64 KiB),
// two workgroups per CU.  64: four stages (64 KiB); such launches are latency-bound and a deep queue of loads is what helps.
template <bool A_KC, bool B_KC, typename OutT, bool MULTI, int TB, int ST>
__global__ __launch_bounds__(256) void gemm_square_kernel(const GemmSmallArgs args) {
    constexpr int T = TB / 32;  // MFMA tiles per wave and direction
    constexpr int STAGE = 2 * TB * BK;
    __shared__ __attribute__((aligned(1024))) bf16_t smem[ST * STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tile, part;
    tile_and_part(args, tile, part);
    const GemmProblem p = problem_of(args, tile);
    int tm, tn;
    tile_of(tile - p.first, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * TB, n0 = tn * TB;
    const int arow = (wave >> 1) * (TB / 2), brow = (wave & 1) * (TB / 2);
    TileLoader<A_KC, TB, 4, true> la;
    TileLoader<B_KC, TB, 4, true> lb;
    const int64_t a_blk = A_KC ? (int64_t)m0 * p.lda : (int64_t)m0;
    const int64_t b_blk = B_KC ? (int64_t)n0 * p.ldb : (int64_t)n0;
    la.init(lane, wave, p.M - m0, p.lda);
    lb.init(lane, wave, p.N - n0, p.ldb);
    const int64_t astep = A_KC ? BK : (int64_t)BK * p.lda;
    const int64_t bstep = B_KC ? BK : (int64_t)BK * p.ldb;
    int kt0;
    const int nk = share_of(MULTI ? args.seg.nk : (args.K + BK - 1) / BK, part, args.nsplit, kt0);
    auto issue_tile = [&](int t, int stage) {
        const bf16_t *Ab, *Bb;
        int kv;
        t += kt0;
        pick_segment<MULTI>(p.A, p.B, args.K, args.seg, t, kv, Ab, Bb);
        la.issue(la.base(Ab + a_blk + (int64_t)t * astep), smem + stage * STAGE, lane, wave, kv);
        lb.issue(lb.base(Bb + b_blk + (int64_t)t * bstep), smem + stage * STAGE + TB * BK, lane, wave, kv);
    };
    constexpr int NLD = decltype(la)::NI + decltype(lb)::NI;
#pragma unroll
    for (int s = 0; s < ST - 1; ++s)
        if (s < nk) issue_tile(s, s);
    f32x4 acc[T][T];
    zero_acc(acc);
    int stage = 0, free_stage = ST - 1;
    for (int kt = 0; kt < nk; ++kt) {
        if (ST > 2 && kt + ST - 2 < nk) wait_loads<(ST - 2) * NLD>();
        else wait_loads<0>();
        wave_barrier();  // K tile kt is in LDS, and every wave is done with K tile kt - 1, whose stage is refilled now
        if (kt + ST - 1 < nk) issue_tile(kt + ST - 1, free_stage);
        const bf16_t* sA = smem + stage * STAGE;
        const bf16_t* sB = sA + TB * BK;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            bf16x8 fa[T], fb[T];
#pragma unroll
            for (int j = 0; j < T; ++j) fb[j] = sfrag<B_KC, TB>(sB, brow + j * 16, ks, lane);
#pragma unroll
            for (int i = 0; i < T; ++i) fa[i] = sfrag<A_KC, TB>(sA, arow + i * 16, ks, lane);
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
        }
        stage = opaque(stage + 1 == ST ? 0 : stage + 1);
        free_stage = free_stage + 1 == ST ? 0 : free_stage + 1;
    }
    if (args.nsplit > 1) store_partial<T, T, TB, TB>(acc, args, tile, part, arow, brow, lane);
    else store_tile<A_KC && B_KC, T, T, OutT>(acc, p, m0, n0, arow, brow, lane);
}

// =================================================================================================
// 64 x 64 tile, the reduction dealt to the 8 waves of a workgroup
// =================================================================================================
// Few tiles and a long reduction (a weight gradient of a narrow layer): each wave multiplies the whole tile over every eighth
// K tile out of its own 16 KiB of LDS, with no barrier in the loop, so eight K tiles are in flight per workgroup; the eight
// sums are added in wave order at the end.
template <bool A_KC, bool B_KC, typename OutT, bool MULTI>
__global__ __launch_bounds__(512) void gemm_64_waves_kernel(const GemmSmallArgs args) {
    constexpr int NW = 8, STAGE = 2 * 64 * BK;
    __shared__ __attribute__((aligned(1024))) bf16_t smem[NW * STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tile, part;
    tile_and_part(args, tile, part);
    const GemmProblem p = problem_of(args, tile);
    int tm, tn;
    tile_of(tile - p.first, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * 64, n0 = tn * 64;
    TileLoader<A_KC, 64, 1, true> la;
    TileLoader<B_KC, 64, 1, true> lb;
    const int64_t a_blk = A_KC ? (int64_t)m0 * p.lda : (int64_t)m0;
    const int64_t b_blk = B_KC ? (int64_t)n0 * p.ldb : (int64_t)n0;
    la.init(lane, 0, p.M - m0, p.lda);
    lb.init(lane, 0, p.N - n0, p.ldb);
    const int64_t astep = A_KC ? BK : (int64_t)BK * p.lda;
    const int64_t bstep = B_KC ? BK : (int64_t)BK * p.ldb;
    const int nk = MULTI ? args.seg.nk : (args.K + BK - 1) / BK;
    auto issue_tile = [&](int t) {
        const bf16_t *Ab, *Bb;
        int kv;
        pick_segment<MULTI>(p.A, p.B, args.K, args.seg, t, kv, Ab, Bb);
        la.issue(la.base(Ab + a_blk + (int64_t)t * astep), smem + wave * STAGE, lane, 0, kv);
        lb.issue(lb.base(Bb + b_blk + (int64_t)t * bstep), smem + wave * STAGE + 64 * BK, lane, 0, kv);
    };
    f32x4 acc[4][4];
    zero_acc(acc);
    if (wave < nk) issue_tile(wave);
    for (int kt = wave; kt < nk; kt += NW) {
        wait_loads<0>();
        __builtin_amdgcn_sched_barrier(0);
        const bf16_t* sA = smem + opaque(wave * STAGE);
        const bf16_t* sB = sA + 64 * BK;
        bf16x8 fa[2][4], fb[2][4];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
            for (int j = 0; j < 4; ++j) fb[ks][j] = sfrag<B_KC, 64>(sB, j * 16, ks, lane);
#pragma unroll
            for (int i = 0; i < 4; ++i) fa[ks][i] = sfrag<A_KC, 64>(sA, i * 16, ks, lane);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the fragments are in registers, the tiles may be overwritten
        __builtin_amdgcn_sched_barrier(0);
        if (kt + NW < nk) issue_tile(kt + NW);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[ks][j], fa[ks][i], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
    float* f = reinterpret_cast<float*>(smem);  // [wave][16 MFMA tiles][64 lanes][4]
    static_assert(NW * 16 * 64 * 4 * 4 <= NW * STAGE * 2, "the sums fit the tile memory");
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4*>(f + ((wave * 16 + i * 4 + j) * 64 + lane) * 4) = acc[i][j];
    __syncthreads();
    f32x4 sum[1][2];  // a wave finishes two neighbouring MFMA tiles: 16 rows x 32 columns
    zero_acc(sum);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(f + ((w * 16 + wave * 2 + q) * 64 + lane) * 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[0][q][r] += x[r];
        }
    store_tile<A_KC && B_KC, 1, 2, OutT>(sum, p, m0, n0, (wave >> 1) * 16, (wave & 1) * 32, lane);
}

// C tile (=|+=) sum of the nsplit fp32 partial tiles, added in index order; a thread owns 8 consecutive columns of one row
template <typename OutT>
__global__ __launch_bounds__(256) void small_reduce_kernel(const GemmSmallArgs args, int tbm, int tbn, int first_tile) {
    const int per_tile = tbm * tbn / 2048;  // workgroups per tile
    const int local = blockIdx.x / per_tile, tile = first_tile + local;
    const GemmProblem p = problem_of(args, tile);
    int tm, tn;
    tile_of(tile - p.first, p.tiles_m, p.tiles_n, tm, tn);
    const int e = ((blockIdx.x - local * per_tile) * 256 + threadIdx.x) * 8;  // element of the tile
    const int rl = e / tbn, cl = e - rl * tbn;
    const int row = tm * tbm + rl, col = tn * tbn + cl;
    if (row >= p.M || col >= p.N) return;
    float v[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = 0.f;
    const size_t stride = (size_t)tbm * tbn;
    const float* src = args.partial + (size_t)local * args.nsplit * stride + e;
#pragma unroll 4
    for (int q = 0; q < args.nsplit; ++q, src += stride) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(src), y = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) { v[r] += x[r]; v[4 + r] += y[r]; }
    }
    if (p.accumulate & kRoundResult) {
#pragma unroll
        for (int r = 0; r < 8; ++r) v[r] = (float)(bf16_t)v[r];
    }
    const bool accumulate = p.accumulate & 1;
    OutT* dst = (OutT*)p.C + (int64_t)row * p.ldc + col;
    if (!vector_stores<OutT>(p)) {
#pragma unroll
        for (int r = 0; r < 8; ++r)
            if (col + r < p.N) dst[r] = (OutT)(accumulate ? v[r] + (float)dst[r] : v[r]);
    } else if constexpr (sizeof(OutT) == 2) {
        if (accumulate) {
            const bf16x8 old = ld_bf16x8((const bf16_t*)dst);
#pragma unroll
            for (int r = 0; r < 8; ++r) v[r] += (float)old[r];
        }
        st_bf16x8((bf16_t*)dst, pack8(v));
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            f32x4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = v[4 * h + r];
            if (accumulate) o += *reinterpret_cast<const f32x4*>(dst + 4 * h);
            *reinterpret_cast<f32x4*>(dst + 4 * h) = o;
        }
    }
}

template <bool A_KC, bool B_KC, typename OutT, bool MULTI>
void launch_kind(int kind, const GemmSmallArgs& a, bool tail, hipStream_t st) {
    const dim3 grid((unsigned)(a.ntiles * a.nsplit));
    switch (kind) {
#define EZL_WIDE(BM_, BN_)                                                                                                                 \
    if (tail) hipLaunchKernelGGL((gemm_wide_kernel<A_KC, B_KC, OutT, MULTI, true, BM_, BN_>), grid, dim3(256), 0, st, a);                  \
    else hipLaunchKernelGGL((gemm_wide_kernel<A_KC, B_KC, OutT, MULTI, false, BM_, BN_>), grid, dim3(256), 0, st, a);                      \
    break
        case kTile256x128: EZL_WIDE(256, 128);
        case kTile192x128: EZL_WIDE(192, 128);
#undef EZL_WIDE
        case kTile128: hipLaunchKernelGGL((gemm_square_kernel<A_KC, B_KC, OutT, MULTI, 128, 2>), grid, dim3(256), 0, st, a); break;
        case kTile64: hipLaunchKernelGGL((gemm_square_kernel<A_KC, B_KC, OutT, MULTI, 64, 4>), grid, dim3(256), 0, st, a); break;
        default: hipLaunchKernelGGL((gemm_64_waves_kernel<A_KC, B_KC, OutT, MULTI>), grid, dim3(512), 0, st, a); break;
    }
    if (a.nsplit > 1) {
        const int tbm = (int)gemm_kind_bm(kind), tbn = (int)gemm_kind_bn(kind);
        hipLaunchKernelGGL((small_reduce_kernel<OutT>), dim3((unsigned)(a.ntiles * (tbm * tbn / 2048))), dim3(256), 0, st, a, tbm, tbn, 0);
    }
}

}  // namespace

void gemm_tile_grids(const GemmPlan& plan, GemmSmallArgs& a, int count) {
    const int bm = (int)gemm_kind_bm(plan.kind), bn = (int)gemm_kind_bn(plan.kind);
    a.ntiles = 0;
    for (int i = 0; i < kMaxProblems; ++i) {
        GemmProblem& p = a.p[i];
        if (i >= count) {
            a.first[i] = 0x7fffffff;
            continue;
        }
        p.tiles_m = (p.M + bm - 1) / bm;
        p.tiles_n = (p.N + bn - 1) / bn;
        p.first = a.first[i] = a.ntiles;
        a.ntiles += p.tiles_m * p.tiles_n;
    }
    a.nsplit = plan.nsplit;
}

void gemm_small_reduce(int kind, bool fp32, int first_tile, const GemmSmallArgs& a, hipStream_t stream) {
    const int bm = (int)gemm_kind_bm(kind), bn = (int)gemm_kind_bn(kind);
    const dim3 grid((unsigned)((a.ntiles - first_tile) * (bm * bn / 2048)));
    if (fp32) hipLaunchKernelGGL((small_reduce_kernel<float>), grid, dim3(256), 0, stream, a, bm, bn, first_tile);
    else hipLaunchKernelGGL((small_reduce_kernel<bf16_t>), grid, dim3(256), 0, stream, a, bm, bn, first_tile);
}

void gemm_small_launch(int form, bool multi, const GemmPlan& plan, GemmSmallArgs& a, int count, hipStream_t stream) {
    gemm_tile_grids(plan, a, count);
    bool tail = a.K % BK != 0;
    if (multi) tail = tail || a.seg.K1 % BK != 0 || a.seg.K2 % BK != 0;
    if (form == 0) launch_kind<true, true, bf16_t, false>(plan.kind, a, tail, stream);
    else if (form == 1 && multi) launch_kind<true, false, bf16_t, true>(plan.kind, a, tail, stream);
    else if (form == 1) launch_kind<true, false, bf16_t, false>(plan.kind, a, tail, stream);
    else if (form == 4) launch_kind<true, true, float, false>(plan.kind, a, tail, stream);
    else if (form == 2) launch_kind<false, false, float, false>(plan.kind, a, tail, stream);
    else launch_kind<false, false, bf16_t, false>(plan.kind, a, tail, stream);
}
