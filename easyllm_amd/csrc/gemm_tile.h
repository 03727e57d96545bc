// Device code shared by the GEMM kernels (gemm.hip, gemm_small.hip): operand tiles in LDS, MFMA fragments, K segments.
#pragma once
#include "common.h"

#include <type_traits>

// MULTI: the reduction runs over up to three (A, B) pairs in turn, C (=|+=) A0 B0 + A1 B1 + A2 B2, all pairs with the same
// leading dimensions: the input gradient of several linears that share their input (q / k / v, gate / up) in one launch,
// summed in fp32, instead of one launch per pair that reads and rewrites the bf16 result.  The kernel's K is pair 0's
// length; pair 1 starts at K tile t1, pair 2 at t2 (nk when absent), nk tiles in all.
struct KSegments {
    const bf16_t* A1;
    const bf16_t* B1;
    const bf16_t* A2;
    const bf16_t* B2;
    int t1, t2, nk;
    int K1, K2;
};

// Kernels take it in the bits of `accumulate`: the product is rounded to bf16 first (logits that are handed out in fp32; with bit 0, a forward product
// added to a bf16 tensor as a launch of its own would add the two).
constexpr int kRoundResult = 2;

namespace {

constexpr int BM = 256, BN = 256, BK = 64;

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
typedef __attribute__((address_space(3))) void lds_void;

// tile id (in the banded order described above) -> tile coordinates
__device__ __forceinline__ void tile_of(int pid, int tiles_m, int tiles_n, int& tm, int& tn) {
    constexpr int GROUP_M = 8;
    const int group_size = GROUP_M * tiles_n;
    const int group = pid / group_size;
    const int first_m = group * GROUP_M;
    const int gm = tiles_m - first_m < GROUP_M ? tiles_m - first_m : GROUP_M;
    tm = first_m + (pid % group_size) % gm;
    tn = (pid % group_size) / gm;
}

// chunk (16 B) permutation of a k-major tile row: keeps the transpose reads of one wave instruction (four k rows x 32 B in each
// of four k octets) on distinct banks.  Rows of 128 or 256 columns all start at bank 0; a row of 64 (192) columns is half (one and a
// half times) the banks wide, so the row's parity already separates two of the four rows.
template <int R>
__device__ __forceinline__ int kmajor_swizzle(int krow) {
    if (R % 128 == 0) return ((krow & 3) << 2) ^ (((krow >> 3) & 1) << 1);
    return (((krow >> 1) & 1) << 2) ^ (((krow >> 3) & 1) << 1);
}

// One operand tile of R rows (k-contiguous) or columns (k-major) = R / 8 wave-instructions of 1 KiB each
// (buffer_load_dwordx4 ... lds: lane l lands at base + 16 l).
//   k-contiguous tile [R rows][64 k]:  instruction q covers rows 8q..8q+7; chunk c of row r sits in slot c ^ ((r>>1)&7)
//   k-major tile      [64 k][R cols]:  instruction q covers 512 / R k rows (not whole ones with R = 192); chunk c of k row sits in slot
//                                      c ^ kmajor_swizzle(k)
// Wave w issues instructions q = w*NI .. w*NI+NI-1, i.e. one contiguous NI KiB piece of the tile: M0 (the LDS base) is
// written once per 4 KiB and the instruction offset (i & 3) * 1024 selects the KiB.  That offset is also added to the global
// address, so the per-lane byte offsets are stored with it already subtracted; they are kept 4 KiB high (and the
// buffer's base 4 KiB low) so that they stay non-negative.  The address is buffer base (scalar, advanced per K tile) +
// 32-bit lane offset + immediate: no vector address arithmetic inside the K loop.
// The buffer form of the load is used rather than the global one because the compiler books a global load to LDS as a
// flat access that may touch both memories, and while one is in flight it turns every counted wait on the LDS fragment
// reads into a full drain (lgkmcnt(0)); with buffer loads the waits inside the K loop are exact counts.
constexpr uint32_t kBufBytes = 0x80000000u;  // every tile is addressed as a 2 GiB buffer: an offset of kBufBytes reads as zero

template <bool KC, int R, int NW, bool KTAIL>
struct TileLoader {
    static constexpr int NI = R / 8 / NW;
    static constexpr int CPR = R / 8;       // k-major: chunks per k row
    uint32_t off[NI];  // byte offsets from (operand base + k advance - 4096)
    // k-major: k row and place in it of a lane's chunk of wave load I.  Where wave loads are whole k rows these are sums of a part of the
    // wave's and one of the lane's alone; dividing the chunk's number instead cost products with a K tail a tenth (weight gradient 7120 x 1336 x 2008
    // 52 -> 57 us, 2048 tokens 48 both ways).
    static_assert(KC || NI * 64 % CPR == 0, "a wave's piece of the tile is whole k rows");
    static __device__ __forceinline__ int k_row(int wave, int i, int lane) {
        if constexpr (64 % CPR == 0) return (64 / CPR) * (wave * NI + i) + lane / CPR;
        else return wave * (NI * 64 / CPR) + (int)((unsigned)(i * 64 + lane) / CPR);
    }
    static __device__ __forceinline__ int k_chunk(int i, int lane) {
        if constexpr (64 % CPR == 0) return lane % CPR;
        else return (int)((unsigned)(i * 64 + lane) % CPR);
    }
    // dim: rows (columns) of the operand from this tile's first on; those past the edge re-read the last one, their results
    // are never stored
    __device__ __forceinline__ void init(int lane, int wave, int dim, int64_t ld) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int q = wave * NI + i;
            int64_t e;
            if (KC) {
                const int row = 8 * q + (lane >> 3);
                const int c = (lane & 7) ^ ((row >> 1) & 7);
                const int gr = row < dim ? row : dim - 1;
                e = (int64_t)gr * ld + c * 8;
            } else {
                const int krow = k_row(wave, i, lane);
                const int c = k_chunk(i, lane) ^ kmajor_swizzle<R>(krow);
                int col = c * 8;
                col = col + 8 <= dim ? col : dim - 8;
                e = (int64_t)krow * ld + col;
            }
            off[i] = (uint32_t)(e * 2 + 4096 - (i & 3) * 1024);
        }
    }
    // gtile: the operand advanced to the tile's first k
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t base(const bf16_t* gtile) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(gtile)) - 4096, 0, kBufBytes, 0x00020000);
    }
    // kv: how many of the tile's 64 k exist (looked at with KTAIL only; more than 64 is fine)
    template <int I>
    __device__ __forceinline__ void issue_at(__amdgpu_buffer_rsrc_t g, bf16_t* stage, int lane, int wave, int kv) const {
        uint32_t o = off[I];
        if (KTAIL && kv < BK) {
            const int q = wave * NI + I;
            const int k = KC ? ((lane & 7) ^ (((8 * q + (lane >> 3)) >> 1) & 7)) * 8 : k_row(wave, I, lane);
            o = k < kv ? o : kBufBytes;
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(g, (lds_void*)(stage + wave * (NI * 512) + (I >> 2) * 2048), 16, o, 0, (I & 3) * 1024, 0);
    }
    template <int I = 0>
    __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t g, bf16_t* stage, int lane, int wave, int kv) const {
        if constexpr (I < NI) {
            issue_at<I>(g, stage, lane, wave, kv);
            issue<I + 1>(g, stage, lane, wave, kv);
        }
    }
};

// ---- LDS -> MFMA 16x16x32 operand fragment: 16 rows (or columns) x 32 k; lane l holds row l & 15, k = 8 (l >> 4) + 0..7 ----
template <bool KC, int R>
__device__ __forceinline__ bf16x8 sfrag(const bf16_t* __restrict__ s, int row0, int ks, int lane) {
    if (KC) {
        const int row = row0 + (lane & 15);
        const int c = (ks * 4 + (lane >> 4)) ^ ((row >> 1) & 7);
        return *reinterpret_cast<const bf16x8*>(s + row * 64 + c * 8);
    } else {
        // a 16-lane group reads an 8(k) x 16(row) block as two 4 x 16 transpose reads; lane i of the group receives column i
        const int krow = ks * 32 + (lane >> 4) * 8 + ((lane & 15) >> 2);
        const int col = row0 + ((lane & 3) << 2);
        const int c = (col >> 3) ^ kmajor_swizzle<R>(krow);
        const bf16_t* p = s + krow * R + c * 8 + (col & 7);
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(p));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(p + 4 * R));  // k + 4: same swizzle
        bf16x8 v;
        v[0] = lo[0]; v[1] = lo[1]; v[2] = lo[2]; v[3] = lo[3];
        v[4] = hi[0]; v[5] = hi[1]; v[6] = hi[2]; v[7] = hi[3];
        return v;
    }
}

// The fragments of a wave's half of a tile's rows (columns), R in all.  What a fragment's address is made of per lane is computed once and hidden
// from the compiler, which otherwise rebuilds it per read in a loop over stages (48 vector instructions per K tile of the 4-wave
// kernel, 5 % of its time); the rest is the read's immediate offset.
template <bool KC, int R>
struct FragReader {
    static constexpr int NF = R / 32;
    int off[KC ? 2 : NF];  // elements: k-contiguous per k half, k-major per fragment (its chunk permutation mixes with the fragment's index)
    __device__ __forceinline__ void init(int row0, int lane) {
        if constexpr (KC) {
            const int row = row0 + (lane & 15);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) off[ks] = row * 64 + (((ks * 4 + (lane >> 4)) ^ ((row >> 1) & 7)) * 8);
        } else {
            const int krow = (lane >> 4) * 8 + ((lane & 15) >> 2);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const int col = row0 + f * 16 + ((lane & 3) << 2);
                off[f] = krow * R + ((col >> 3) ^ kmajor_swizzle<R>(krow)) * 8 + (col & 7);
            }
        }
#pragma unroll
        for (int& o : off) asm volatile("" : "+v"(o));
    }
    template <int F>
    __device__ __forceinline__ bf16x8 read(const bf16_t* __restrict__ s, int ks) const {
        if constexpr (KC) {
            return *reinterpret_cast<const bf16x8*>(s + off[ks] + F * 16 * 64);
        } else {
            const bf16_t* p = s + off[F] + ks * 32 * R;
            const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(p));
            const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(p + 4 * R));
            bf16x8 v;
            v[0] = lo[0]; v[1] = lo[1]; v[2] = lo[2]; v[3] = lo[3];
            v[4] = hi[0]; v[5] = hi[1]; v[6] = hi[2]; v[7] = hi[3];
            return v;
        }
    }
};

// the (A, B) pair of K tile t, the tile's index inside it and how many of its 64 k exist: scalar selects
template <bool MULTI>
__device__ __forceinline__ void pick_segment(const bf16_t* A, const bf16_t* B, int K, const KSegments& seg, int& t, int& kv,
                                             const bf16_t*& Ab, const bf16_t*& Bb) {
    Ab = A;
    Bb = B;
    if constexpr (MULTI) {
        const bool s1 = t >= seg.t1, s2 = t >= seg.t2;
        Ab = s2 ? seg.A2 : (s1 ? seg.A1 : A);
        Bb = s2 ? seg.B2 : (s1 ? seg.B1 : B);
        t -= s2 ? seg.t2 : (s1 ? seg.t1 : 0);
        K = s2 ? seg.K2 : (s1 ? seg.K1 : K);
    }
    kv = K - t * BK;
}

// A barrier that waits for nothing: what is in flight is each wave's to wait for first, by a count.  (In front of a __syncthreads the
// compiler puts a wait for all loads that go straight to LDS, those of later K tiles included.)
__device__ __forceinline__ void wave_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
}

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// Tiles of 48 accumulators and more are the 4-wave kernel's, which lie in AGPRs: they are copied out here, row by row (with a
// scheduling barrier behind each).  Copied any earlier, behind their MFMA or all of them before the first store, they spill.
template <int ACCUMULATORS>
__device__ __forceinline__ f32x4 from_agprs(f32x4 x) {
    if constexpr (ACCUMULATORS >= 48) asm volatile("" : "+a"(x));
    return x;
}

// acc[i][j] register r is C[m0 + row0 + 16 i + (lane & 15)][n0 + col0 + 16 j + 4 (lane >> 4) + r].
// C is addressed as a buffer that starts at the tile's corner and ends behind the last valid element of its last valid row: a
// store past either edge drops out by the range check (for columns: an offset that is out of range), so the code is
// straight-line (a branch per store instead: 4000 x 32000 x 2048 with an fp32 result 632 us against 482; a weight gradient of
// 32000 x 4096 over 1531 tokens 420 against 405).  bf16: lanes l and l ^ 16 trade halves of two neighbouring column tiles, 16-byte stores.  VEC = false (rows
// that do not start on 16 bytes, or a width that is no multiple of 8): one element per store.
// A row's old values (ACC) are fetched in front of the stores of the row before it: an access waits for all older ones.
// The row step is part of the vector offset: with a scalar offset register the compiler leaves no wait state between a 16-byte
// buffer store and the next write of its data registers, and the hardware needs one (seen as lanes 12 - 15 of a row group holding
// the next value's bits where such a write came right behind).
template <int TM, int TN, typename OutT, bool ACC, bool VEC, bool ROUND = false>
__device__ __forceinline__ void store_tile_impl(const f32x4 (&acc)[TM][TN], OutT* C, int64_t ldc, int mrem, int nrem, int row0, int col0,
                                                int lane) {
    constexpr int SZ = (int)sizeof(OutT);
    constexpr uint32_t kOut = 0x80000000u;
    const __amdgpu_buffer_rsrc_t cbuf = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<char*>(C), 0, (uint32_t)(((int64_t)(mrem - 1) * ldc + nrem) * SZ), 0x00020000);
    const uint32_t row_off = (uint32_t)(row0 + (lane & 15)) * (uint32_t)(ldc * SZ);
    const uint32_t row_step = (uint32_t)(16 * ldc * SZ);
    if constexpr (!VEC) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int col = col0 + j * 16 + 4 * (lane >> 4) + r;
                    const uint32_t voff = col < nrem ? row_off + (uint32_t)col * SZ : kOut;
                    float v = acc[i][j][r];
                    if constexpr (ROUND) v = (float)(bf16_t)v;
                    if constexpr (SZ == 2) {
                        if constexpr (ACC) v += (float)__builtin_bit_cast(bf16_t, __builtin_amdgcn_raw_buffer_load_b16(cbuf, voff + i * row_step, 0, 0));
                        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, (bf16_t)v), cbuf, voff + i * row_step, 0, 0);
                    } else {
                        if constexpr (ACC) v += __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(cbuf, voff + i * row_step, 0, 0));
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), cbuf, voff + i * row_step, 0, 0);
                    }
                }
    } else if constexpr (SZ == 2) {
        const int g = lane >> 4;
        const auto offset = [&](int jp) {
            const int col = col0 + (2 * jp + (g & 1)) * 16 + 8 * (g >> 1);
            return col < nrem ? row_off + (uint32_t)col * SZ : kOut;
        };
        u32x4 old[2][TN / 2];
        const auto fetch = [&](int i) {
#pragma unroll
            for (int jp = 0; jp < TN / 2; ++jp) old[i & 1][jp] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(cbuf, offset(jp) + i * row_step, 0, 0));
        };
        if constexpr (ACC) fetch(0);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if constexpr (ACC)
                if (i + 1 < TM) fetch(i + 1);
#pragma unroll
            for (int jp = 0; jp < TN / 2; ++jp) {
                const f32x4 va = from_agprs<TM * TN>(acc[i][2 * jp]), vb = from_agprs<TM * TN>(acc[i][2 * jp + 1]);
                float v[8];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(va[r]), __float_as_uint(vb[r]), false, false);
                    v[r] = __uint_as_float(sw[0]);
                    v[4 + r] = __uint_as_float(sw[1]);
                }
                if constexpr (ACC) {
                    const bf16x8 o = __builtin_bit_cast(bf16x8, old[i & 1][jp]);
#pragma unroll
                    for (int r = 0; r < 8; ++r) v[r] = (ROUND ? (float)(bf16_t)v[r] : v[r]) + (float)o[r];
                }
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, pack8(v)), cbuf, offset(jp) + i * row_step, 0, 0);
            }
            if constexpr (TM * TN >= 48) __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        const auto offset = [&](int j) {
            const int col = col0 + j * 16 + 4 * (lane >> 4);
            return col < nrem ? row_off + (uint32_t)col * SZ : kOut;
        };
        u32x4 old[2][TN];
        const auto fetch = [&](int i) {
#pragma unroll
            for (int j = 0; j < TN; ++j) old[i & 1][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(cbuf, offset(j) + i * row_step, 0, 0));
        };
        if constexpr (ACC) fetch(0);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if constexpr (ACC)
                if (i + 1 < TM) fetch(i + 1);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f32x4 v = from_agprs<TM * TN>(acc[i][j]);
                if constexpr (ROUND)
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = (float)(bf16_t)v[r];
                if constexpr (ACC) {
                    const f32x4 o = __builtin_bit_cast(f32x4, old[i & 1][j]);
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] += o[r];
                }
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), cbuf, offset(j) + i * row_step, 0, 0);
            }
            if constexpr (TM * TN >= 48) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// as above with the kernel's flags: bit 0 accumulate, kRoundResult (only where the form has it: MAY_ROUND; an fp32 result has it without bit 0, a bf16
// one, which is rounded as it is stored, with it)
template <int TM, int TN, typename OutT, bool VEC, bool MAY_ROUND>
__device__ __forceinline__ void store_tile_flags(const f32x4 (&acc)[TM][TN], OutT* C, int64_t ldc, int mrem, int nrem, int row0, int col0,
                                                 int lane, int flags) {
    if (MAY_ROUND && sizeof(OutT) == 2 && flags == (1 | kRoundResult)) store_tile_impl<TM, TN, OutT, true, VEC, MAY_ROUND && sizeof(OutT) == 2>(acc, C, ldc, mrem, nrem, row0, col0, lane);
    else if (flags & 1) store_tile_impl<TM, TN, OutT, true, VEC>(acc, C, ldc, mrem, nrem, row0, col0, lane);
    else if (MAY_ROUND && sizeof(OutT) == 4 && (flags & kRoundResult)) store_tile_impl<TM, TN, OutT, false, VEC, true>(acc, C, ldc, mrem, nrem, row0, col0, lane);
    else store_tile_impl<TM, TN, OutT, false, VEC>(acc, C, ldc, mrem, nrem, row0, col0, lane);
}

}  // namespace

// One product of a launch of the smaller-tile kernels (gemm_small.hip).
struct GemmProblem {
    const bf16_t* A;
    const bf16_t* B;
    void* C;
    int64_t lda, ldb, ldc;
    int M, N;
    int tiles_m, tiles_n, first;  // tile grid, and the launch-wide id of its first tile
    int accumulate;
};

// A launch: independent products over the same K (up to the seven weight gradients of a decoder layer), or (K segments) one
// product over up to three operand pairs.
constexpr int kMaxProblems = 7;
struct GemmSmallArgs {
    GemmProblem p[kMaxProblems];
    int first[kMaxProblems];  // as in p (INT_MAX: no such product), together: one scalar load brings all of them
    int ntiles, K, nsplit;
    float* partial;  // nsplit > 1: [ntiles][nsplit][tile] fp32
    KSegments seg;
};

// Tile shapes: the first two of gemm.hip, the others of gemm_small.hip.
enum GemmKind { kTile256 = 0, kTile192x256, kTile256x128, kTile192x128, kTile128, kTile64, kTile64Waves, kGemmKinds };
constexpr int kKindRows[kGemmKinds] = {256, 192, 256, 192, 128, 64, 64}, kKindCols[kGemmKinds] = {256, 256, 128, 128, 128, 64, 64};
inline bool gemm_kind_large(int kind) { return kind <= kTile192x256; }
struct GemmPlan {
    int kind, nsplit;
};
// form 0: A, B k-contiguous, bf16 result; 1: A k-contiguous, bf16 result (multi: over K segments); 2 / 3: neither, fp32 / bf16
// result; 4: as 0 with an fp32 result.  Sets the tile grids in `a` and launches; 256 rows of every problem's C must span less than 2 GiB.
__attribute__((visibility("hidden"))) void gemm_small_launch(int form, bool multi, const GemmPlan& plan, GemmSmallArgs& a, int count,
                                                             hipStream_t stream);
// tile grids of a launch on tiles of that plan's shape (K is set)
__attribute__((visibility("hidden"))) void gemm_tile_grids(const GemmPlan& plan, GemmSmallArgs& a, int count);
// results (fp32, else bf16) of tiles first_tile.. of a launch from their partial tiles (a.partial: of first_tile on, a.nsplit of each)
__attribute__((visibility("hidden"))) void gemm_small_reduce(int kind, bool fp32, int first_tile, const GemmSmallArgs& a, hipStream_t stream);
inline int64_t gemm_kind_bm(int kind) { return kKindRows[kind]; }
inline int64_t gemm_kind_bn(int kind) { return kKindCols[kind]; }
