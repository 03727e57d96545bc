// Device code shared by the attention kernels (attention.hip, attention_small.hip): parameters, work list, LDS tiles, fragments.
#pragma once
#include "common.h"

#include <type_traits>

struct AttnParams {
    const bf16_t* q; const bf16_t* k; const bf16_t* v; const bf16_t* o; const bf16_t* dout;
    bf16_t* out; bf16_t* dq; bf16_t* dk; bf16_t* dv;
    float* lse; float* delta;
    float* part;  // dK/dV kernel with nsplit > 1: fp32 partial sums [nsplit][2 (dK, dV)][T][nk][d]
    int nsplit;   // workgroups that share a (kv head, key block): each takes nq / nk / nsplit of the group's query heads
    const int* cu;
    int ndocs, s_len, T, nq, nk;
    float scale;
    int64_t q_ss, q_sb, k_ss, k_sb, v_ss, v_sb, o_ss, o_sb;          // forward tensors
    int64_t do_ss, do_sb, dq_ss, dq_sb, dk_ss, dk_sb, dv_ss, dv_sb;  // backward tensors
};

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
typedef __attribute__((address_space(3))) void lds_void;


__device__ __forceinline__ int64_t tok_off(int n, int s_len, int64_t ss, int64_t sb) {
    const int b = n / s_len;
    return (int64_t)b * sb + (int64_t)(n - b * s_len) * ss;
}

// Work list of the three kernels.  A document is cut at batch-row boundaries (the reference's collator never emits one
// that crosses a row: it appends every row's length to that row's boundaries), so inside a piece token i lives at
// tok_off(piece_start) + i * seq_stride and no per-token division is needed.  A piece of n tokens has ceil(n / 128) blocks;
// block j of a piece (queries, or keys counted from the piece's END for the dK/dV kernel) walks j + 1 blocks of the other
// operand, so its running time grows with j.
//
// Blocks are handed out longest first over ALL pieces and heads (rank 0 = the largest j anywhere): the hardware starts
// workgroups in the order of their ids, and with the long blocks of some head started late -- as happens when ids run head
// by head -- the last of them finish long after everything else (98 instead of 66 block-times for 4 heads x 32 blocks on
// the 64 slots of an XCD).  rank -> (piece, j): level j holds the pieces with more than j blocks, levels are laid out from
// the highest down; the level is found by bisection on count(j) = number of blocks with index >= j, the piece inside the
// level by a prefix sum, both computed by the whole workgroup (every thread must call this, before any other use of LDS).
// Dense batches (no cu_seqlens) have a closed form.
__device__ __forceinline__ int doc_bounds(const int* __restrict__ cu, int d, int s_len, int T, int& e) {
    int a = cu ? cu[d] : d * s_len;
    e = cu ? cu[d + 1] : (d + 1) * s_len;
    a = a < 0 ? 0 : a;
    e = e > T ? T : e;
    return a;
}

struct BlockSearch {
    int* s_wave;  // [16]
    int tid, nthr, lane, wv, nwaves;
    // sum over the workgroup; uniform result
    __device__ __forceinline__ int reduce(int v) const {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        __syncthreads();  // s_wave of the previous reduction has been read
        if (lane == 0) s_wave[wv] = v;
        __syncthreads();
        int t = 0;
        for (int i = 0; i < nwaves; ++i) t += s_wave[i];
        return t;
    }
};

// lds: kFindBlockInts ints of LDS for the search.  It is handed in by the kernel, carved from its one LDS array, instead of
// being declared here: with several LDS variables in a kernel the compiler tags every LDS access with the variable it
// belongs to and thereby drops the no-alias tags of the fragment reads, after which each read waits for all tile loads in
// flight (vmcnt(0)) because it might alias their destination.
constexpr int kFindBlockInts = 20;
__device__ __forceinline__ bool find_block(const int* __restrict__ cu, int ndocs, int s_len, int T, int rank, int blk_rows,
                                           int& doc_start, int& doc_len, int& blk, int* lds) {
    const int nb_row = (s_len + blk_rows - 1) / blk_rows;
    if (!cu) {  // every piece is a whole batch row: level j holds all ndocs rows
        if (rank >= ndocs * nb_row) return false;
        blk = nb_row - 1 - rank / ndocs;
        doc_start = (rank % ndocs) * s_len;
        doc_len = s_len;
        return true;
    }
    int* s_wave = lds;        // [16]
    int* s_found = lds + 16;  // [4]
    BlockSearch bs;
    bs.s_wave = s_wave;
    bs.tid = threadIdx.x; bs.nthr = blockDim.x; bs.lane = bs.tid & 63; bs.wv = bs.tid >> 6; bs.nwaves = bs.nthr >> 6;
    // blocks with index >= j over this thread's documents (pieces enumerated on the fly; one piece unless a document
    // crosses a batch row)
    auto count_ge = [&](int j) {
        int c = 0;
        for (int d = bs.tid; d < ndocs; d += bs.nthr) {
            int e;
            const int a = doc_bounds(cu, d, s_len, T, e);
            for (int x = a; x < e;) {
                const int row_end = (x / s_len + 1) * s_len;
                const int e1 = e < row_end ? e : row_end;
                const int nb = (e1 - x + blk_rows - 1) / blk_rows;
                c += nb > j ? nb - j : 0;
                x = e1;
            }
        }
        return bs.reduce(c);
    };
    if (rank >= count_ge(0)) return false;
    int lo = 0, hi = nb_row, c_hi = 0;  // count(lo) > rank >= count(hi)
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        const int c = count_ge(mid);
        if (c > rank) lo = mid;
        else { hi = mid; c_hi = c; }
    }
    const int j = lo;
    const int want = rank - c_hi;  // the want-th piece (in document order) that has more than j blocks
    if (bs.tid == 0) s_found[0] = 0;
    int base = 0;
    for (int d0 = 0; d0 < ndocs; d0 += bs.nthr) {
        const int d = d0 + bs.tid;
        int mine = 0, a = 0, e = 0;
        if (d < ndocs) {
            a = doc_bounds(cu, d, s_len, T, e);
            for (int x = a; x < e;) {
                const int row_end = (x / s_len + 1) * s_len;
                const int e1 = e < row_end ? e : row_end;
                mine += (e1 - x + blk_rows - 1) / blk_rows > j;
                x = e1;
            }
        }
        int incl = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (bs.lane >= o) incl += v;
        }
        __syncthreads();
        if (bs.lane == 63) s_wave[bs.wv] = incl;
        __syncthreads();
        int before = 0, total = 0;
        for (int i = 0; i < bs.nwaves; ++i) {
            const int v = s_wave[i];
            before += i < bs.wv ? v : 0;
            total += v;
        }
        const int first = base + before + incl - mine;  // rank inside the level of this thread's first qualifying piece
        if (mine > 0 && want >= first && want < first + mine) {
            int rel = want - first;
            for (int x = a; x < e;) {
                const int row_end = (x / s_len + 1) * s_len;
                const int e1 = e < row_end ? e : row_end;
                if ((e1 - x + blk_rows - 1) / blk_rows > j) {
                    if (rel == 0) {
                        s_found[1] = x;
                        s_found[2] = e1 - x;
                        s_found[0] = 1;
                        break;
                    }
                    --rel;
                }
                x = e1;
            }
        }
        base += total;
        if (want < base) break;  // uniform
    }
    __syncthreads();
    if (!s_found[0]) return false;
    doc_start = __builtin_amdgcn_readfirstlane(s_found[1]);
    doc_len = __builtin_amdgcn_readfirstlane(s_found[2]);
    blk = j;
    return true;
}

// The hardware deals consecutive workgroups (x fastest, then y) round-robin to the 8 XCDs, each with an L2 of its own.
// With the plain (block, head) numbering every XCD would touch the K / V rows of every head and its L2 would keep missing;
// renumbered, an XCD owns nheads / 8 heads, and inside an XCD the ids run over ranks (longest blocks first, see above) with
// the XCD's heads innermost: blocks of equal length of all its heads start together and walk the keys in step.
// by: head, rank: position in the longest-first work list of one head.
// (lin: workgroup number)
__device__ __forceinline__ void heads_of(int lin, int nheads, int& rank, int& by) {
    if ((nheads & 7) == 0) {
        const int hpx = nheads >> 3, idx = lin >> 3;
        by = (lin & 7) * hpx + idx % hpx;
        rank = idx / hpx;
    } else {
        by = lin % nheads;
        rank = lin / nheads;
    }
}
__device__ __forceinline__ void xcd_head_blocks(int nheads, int& rank, int& by) {
    heads_of(blockIdx.y * gridDim.x + blockIdx.x, nheads, rank, by);
}

template <int D>
struct Tile {
    static constexpr int LD = D + 24;             // padded row stride in elements
    static constexpr int CH = D / 8;              // 128-bit chunks per row
    static constexpr int ROWS = 64;
    static constexpr int ELEMS = ROWS * LD;

    // ---- tile rows straight from global memory into LDS (buffer_load ... lds, 16 bytes per lane) ----
    // One wave instruction fills 1 KiB of consecutive LDS, i.e. 1024 / (2 LD) padded rows: instruction q of a tile covers
    // bytes 1024 q .. 1024 q + 1023 of its LDS image, and the lane that falls on row padding re-reads the row's first chunk.
    // Rows at or past the document's end re-read its last row: finite values that only ever meet masked probabilities.
    // NWAVES waves share the NQ instructions of a tile: wave w issues q = w, w + NWAVES, ...
    static constexpr int NQ = (ROWS * LD * 2 + 1023) / 1024;
    static_assert(ROWS * LD * 2 % 1024 == 0, "a tile is a whole number of 1 KiB pieces");
    template <int NWAVES>
    struct Direct {
        static constexpr int NJ = (NQ + NWAVES - 1) / NWAVES;
        uint32_t off[NJ];  // global byte offset of this lane's chunk from the tile's first row, per instruction
        // last: last valid row of the tile (63, or fewer in a document's ragged last tile: later rows re-read it)
        __device__ __forceinline__ void init(int64_t ss, int lane, int wave, int last) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int q = wave + NWAVES * j;
                const int byte = q * 1024 + lane * 16;
                int row = byte / (LD * 2);
                int colb = byte - row * (LD * 2);
                colb = colb < D * 2 ? colb : 0;
                row = row < last ? row : last;
                off[j] = (uint32_t)row * (uint32_t)(ss * 2) + (uint32_t)colb;
            }
        }
        // tile_rows: global address of the tile's first row (head column included); stage: its LDS image
        __device__ __forceinline__ void issue(const bf16_t* tile_rows, bf16_t* stage, int wave) const {
            // (the buffer form of the load: while a global load to LDS is in flight the compiler, which books it as a flat
            // access, turns every counted wait on LDS reads into a full drain)
            const __amdgpu_buffer_rsrc_t g = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<char*>(reinterpret_cast<const char*>(tile_rows)), 0, 0xffffffffu, 0x00020000);
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int q = wave + NWAVES * j;
                if (q < NQ) __builtin_amdgcn_raw_ptr_buffer_load_lds(g, (lds_void*)(stage + q * 512), 16, off[j], 0, 0, 0);
            }
        }
    };
    // operand whose k index is d:   lane -> row (row0 + lane&31), d = kd*16 + 8*(lane>>5) ..+7
    static __device__ __forceinline__ bf16x8 frag_kc(const bf16_t* __restrict__ s, int row0, int kd, int lane) {
        return *reinterpret_cast<const bf16x8*>(s + (row0 + (lane & 31)) * LD + kd * 16 + (lane >> 5) * 8);
    }
    // operand whose k index is the tile row: lane -> d column (col0 + lane&31); k values are tile rows
    // krow0 + 4g + {0..3} and krow0 + 8 + 4g + {0..3}, g = lane>>5 -- the order in which a 32x32
    // accumulator block holds 16 consecutive rows, so accumulators convert straight to the B operand.
    static __device__ __forceinline__ bf16x8 frag_tr(const bf16_t* __restrict__ s, int krow0, int col0, int lane) {
        const int q = lane >> 4;
        const bf16_t* p = s + (krow0 + 4 * (lane >> 5) + ((lane & 15) >> 2)) * LD + col0 + (q & 1) * 16 + ((lane & 3) << 2);
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(p));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(p + 8 * LD));
        bf16x8 v;
        v[0] = lo[0]; v[1] = lo[1]; v[2] = lo[2]; v[3] = lo[3];
        v[4] = hi[0]; v[5] = hi[1]; v[6] = hi[2]; v[7] = hi[3];
        return v;
    }
    // ---- fragments of the 16x16x32 MFMA (l16 = lane & 15, j4 = lane >> 4) ----
    // (the tile pointers are __restrict__ so that the reads carry a no-alias tag: an untagged LDS read waits for every tile
    // load in flight)
    // A operand whose k index is d: 16 tile rows row0 .., d = 32 ds + 8 j4 .. + 7
    static __device__ __forceinline__ bf16x8 frag_kc16(const bf16_t* __restrict__ s, int row0, int ds, int lane) {
        return *reinterpret_cast<const bf16x8*>(s + (row0 + (lane & 15)) * LD + ds * 32 + (lane >> 4) * 8);
    }
    // A operand whose k index is the tile row: lane -> d column col0 + l16; k slots 8 j4 + e are tile rows krow0 + 4 j4 + e
    // (e < 4) and krow0 + 16 + 4 j4 + e - 4 (e >= 4): the order in which two stacked 16-row accumulator tiles hold them
    static __device__ __forceinline__ bf16x8 frag_tr16(const bf16_t* __restrict__ s, int krow0, int col0, int lane) {
        const bf16_t* a = s + (krow0 + 4 * (lane >> 4) + ((lane & 15) >> 2)) * LD + col0 + ((lane & 3) << 2);
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(a));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(a + 16 * LD));
        bf16x8 v;
        v[0] = lo[0]; v[1] = lo[1]; v[2] = lo[2]; v[3] = lo[3];
        v[4] = hi[0]; v[5] = hi[1]; v[6] = hi[2]; v[7] = hi[3];
        return v;
    }
};

// registers 8t .. 8t+7 of an accumulator block as a bf16 B operand
__device__ __forceinline__ bf16x8 acc_to_b(const f32x16& a, int t) {
    bf16x8 v;
    if (t == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (bf16_t)a[e];
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (bf16_t)a[8 + e];
    }
    return v;
}

// row of register r inside a 32-row accumulator block
__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// one operand row per lane, straight from global memory, as D/16 B-operand fragments
template <int D>
__device__ __forceinline__ void load_row_frags(const bf16_t* __restrict__ rowp, int lane, bf16x8* f) {
#pragma unroll
    for (int kd = 0; kd < D / 16; ++kd) f[kd] = *reinterpret_cast<const bf16x8*>(rowp + kd * 16 + (lane >> 5) * 8);
}

// f(integral_constant<int, I>) for I = I0 .. N-1, so that the body sees its index as a constant expression
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

}  // namespace

// Sizes of a call, from which its kernels are chosen.
struct AttnSizes {
    bool documents;  // cu_seqlens given
    int64_t ndocs, total_tokens, s_len, nq, nk, d;
    int64_t rows() const { return total_tokens / s_len; }
    // workgroups of `block` queries or keys per head: as many as any documents can need, hence as many as are launched with documents
    int64_t launched(int64_t block) const { return (total_tokens + block - 1) / block + ndocs + rows(); }
    // documents lie on the device: the host knows how long they are on average, and that none is longer than a batch row
    int64_t mean_length() const {
        const int64_t mean = (total_tokens + ndocs - 1) / ndocs;
        return mean < s_len ? mean : s_len;
    }
};

// attention_small.hip: the same results with 32 queries (or keys) per workgroup
__attribute__((visibility("hidden"))) bool attn_small_pays(const AttnSizes& z, bool backward);
__attribute__((visibility("hidden"))) void attn_small_fwd(const AttnParams& p, int d, hipStream_t stream);
__attribute__((visibility("hidden"))) void attn_small_bwd(const AttnParams& p, int d, hipStream_t stream);
