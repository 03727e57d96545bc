// One decoder layer's forward or backward as a single call: the launches of ParallelTransformerLayer (llama/transformer.py:747-803
// of the reference: RMSNorm, q/k/v, rotary, causal attention, o, add + RMSNorm, gate/up, SwiGLU, down, add) made one after the
// other from native code.
//
// Each of them through the Python wrappers costs the host 10 - 20 us (autograd node, allocation, argument checks), more than a
// small layer's kernels take on the GPU; from here a launch costs the 3 us of the HIP call.  The kernels, their order of
// summation and their results are those of the separate entry points of ezl.h, which this file only calls.
//
// Memory: activations that backward needs lie in one `saved` block, everything else in one `temp` block; both are the caller's
// and laid out by the same arithmetic in forward and backward (bump allocation, 256-byte steps).
#include "common.h"
#include "gemm_list.h"
#include "norm_pair.h"
#include "qkv_bias.h"
#include "../../include/ezl.h"

namespace {

struct Bump {
    char* base;
    int64_t used = 0;
    explicit Bump(void* p) : base((char*)p) {}
    void* take(int64_t bytes) {
        void* p = base ? base + used : nullptr;
        used += (bytes + 255) / 256 * 256;
        return p;
    }
};

struct Dims {
    int64_t T, h, nq, nk, d, f, qw, kw;
    explicit Dims(const ezl_layer& l) : T(l.s * l.b), h(l.h), nq(l.nq), nk(l.nk), d(l.d), f(l.f), qw(l.nq * l.d), kw(l.nk * l.d) {}
};

struct Saved {
    void *n1, *rstd1, *q, *k, *v, *ctx, *lse, *sum, *n2, *rstd2, *gate, *up, *act;
    int64_t bytes;
    Saved(const Dims& m, void* base) {
        Bump b(base);
        n1 = b.take(m.T * m.h * 2); rstd1 = b.take(m.T * 4);
        q = b.take(m.T * m.qw * 2); k = b.take(m.T * m.kw * 2); v = b.take(m.T * m.kw * 2);
        ctx = b.take(m.T * m.qw * 2); lse = b.take(m.nq * m.T * 4);
        sum = b.take(m.T * m.h * 2); n2 = b.take(m.T * m.h * 2); rstd2 = b.take(m.T * 4);
        gate = b.take(m.T * m.f * 2); up = b.take(m.T * m.f * 2); act = b.take(m.T * m.f * 2);
        bytes = b.used;
    }
};

int64_t max64(int64_t a, int64_t b) { return a > b ? a : b; }

// workspace of up to three products over one K, however they are launched
int64_t products_ws(int a_kc, int count, const int64_t* M, const int64_t* N, int64_t K) {
    const int64_t group = count > 1 ? ezl_gemm_group_form_workspace_bytes(a_kc, count, M, N, K) : -1;
    if (group >= 0) return group;
    int64_t w = 0;
    for (int i = 0; i < count; ++i) w = max64(w, ezl_gemm_workspace_bytes(M[i], N[i], K));
    return w;
}

// Sizes of a layer's weight gradients dw_i[n_i, k_i], which all reduce over the T tokens: q, k, v, o, gate, up, down.
struct WeightGradients {
    int64_t n[kGemmListMax], k[kGemmListMax];
    explicit WeightGradients(const Dims& m)
        : n{m.qw, m.kw, m.kw, m.h, m.f, m.f, m.h}, k{m.h, m.h, m.h, m.qw, m.h, m.h, m.f} {}
    // workspace of all of them in one launch behind everything else; -1 where it is faster to launch them as their operands
    // appear (q / k / v, o, gate / up, down).  elem: bytes of a result.  On the smaller tiles, results of much more than the last-level cache (256 MB)
    // are better written in pieces, which drain into memory under the products between them: a layer's backward with 309 and 356 MB of
    // them in one launch and in pieces 301 against 312 us, 1060 against 1102; with 410 - 670 MB 406 against 398, 790 against 779, 968
    // against 1006, 524 against 484, 575 against 534.
    int64_t list_bytes(int64_t T, int elem) const {
        static const int counts[4] = {3, 1, 2, 1};
        int64_t results = 0;
        for (int i = 0; i < kGemmListMax; ++i) results += n[i] * k[i] * elem;
        return gemm_list_workspace_bytes(4, counts, n, k, T, results > (384LL << 20));
    }
};

struct ForwardTemp {
    void *wide, *bias_in, *ws;
    int64_t ws_bytes, bytes;
    ForwardTemp(const ezl_layer& l, const Dims& m, void* base) {
        Bump b(base);
        wide = b.take(m.T * m.h * 2);                                     // o / down result
        bias_in = l.bq ? b.take(m.T * (m.qw + 2 * m.kw) * 2) : nullptr;  // q, k, v before their bias
        const int64_t Tq[3] = {m.T, m.T, m.T}, nqkv[3] = {m.qw, m.kw, m.kw}, ngu[2] = {m.f, m.f};
        ws_bytes = max64(products_ws(1, 3, Tq, nqkv, m.h), products_ws(1, 2, Tq, ngu, m.h));
        ws_bytes = max64(ws_bytes, max64(ezl_gemm_workspace_bytes(m.T, m.h, m.qw), ezl_gemm_workspace_bytes(m.T, m.h, m.f)));
        ws = b.take(ws_bytes);
        bytes = b.used;
    }
};

struct BackwardTemp {
    void *dact, *dgate, *dup, *dn, *dsum, *dctx, *dqkv, *delta, *ln2_sums, *ws;
    int64_t ws_bytes, bytes;
    BackwardTemp(const ezl_layer& l, const Dims& m, void* base) {
        Bump b(base);
        dact = b.take(m.T * m.f * 2); dgate = b.take(m.T * m.f * 2); dup = b.take(m.T * m.f * 2);
        dn = b.take(m.T * m.h * 2); dsum = b.take(m.T * m.h * 2);
        dctx = b.take(m.T * m.qw * 2);
        dqkv = b.take(m.T * (m.qw + 2 * m.kw) * 2);  // dq | dk | dv in one row, so that one launch can reduce over all three
        delta = b.take(m.nq * m.T * 4);
        ln2_sums = b.take(ezl_rmsnorm_bwd_workspace_bytes(m.T, m.h));
        const int64_t mqkv[3] = {m.qw, m.kw, m.kw}, hh[3] = {m.h, m.h, m.h}, mgu[2] = {m.f, m.f};
        int64_t w = max64(products_ws(0, 3, mqkv, hh, m.T), products_ws(0, 2, mgu, hh, m.T));
        w = max64(w, max64(ezl_gemm_workspace_bytes(m.qw, m.h, m.T), ezl_gemm_workspace_bytes(m.f, m.h, m.T)));  // (also one by one)
        w = max64(w, max64(ezl_gemm_workspace_bytes(m.kw, m.h, m.T), ezl_gemm_workspace_bytes(m.h, m.qw, m.T)));
        w = max64(w, max64(ezl_gemm_workspace_bytes(m.h, m.f, m.T), ezl_gemm_workspace_bytes(m.T, m.f, m.h)));
        w = max64(w, max64(ezl_gemm_workspace_bytes(m.T, m.qw, m.h), ezl_gemm_workspace_bytes(m.T, m.h, 2 * m.f)));
        w = max64(w, ezl_gemm_workspace_bytes(m.T, m.h, m.qw + 2 * m.kw));
        w = max64(w, ezl_rmsnorm_bwd_workspace_bytes(m.T, m.h));
        w = max64(w, ezl_attn_bwd_workspace_bytes(m.T, l.ndocs, m.nq, m.nk, m.d));
        if (l.bq) w = max64(w, ezl_bias_grad_workspace_bytes(m.T, m.qw + 2 * m.kw));
        w = max64(w, max64(WeightGradients(m).list_bytes(m.T, 2), WeightGradients(m).list_bytes(m.T, 4)));
        ws_bytes = w;
        ws = b.take(ws_bytes);
        bytes = b.used;
    }
};

#define EZL_TRY(call)                   \
    do {                                \
        if (const int rc__ = (call)) return rc__; \
    } while (0)

// y_i[T, n_i] = x[T, k] w_i[n_i, k]^T
int forward_products(int count, const void* x, const void* const* w, void* const* y, int64_t T, const int64_t* n, int64_t k, void* ws,
                     int64_t ws_bytes, void* st) {
    const int64_t Ts[3] = {T, T, T}, ks[3] = {k, k, k};
    const void* xs[3] = {x, x, x};
    const int zero[3] = {0, 0, 0};
    if (count > 1 && ezl_gemm_group_form_workspace_bytes(1, count, Ts, n, k) >= 0)
        return ezl_gemm_bf16_group(count, xs, w, y, Ts, n, k, ks, ks, n, 1, 1, 0, zero, ws, ws_bytes, st);
    for (int i = 0; i < count; ++i) EZL_TRY(ezl_gemm_bf16(x, w[i], y[i], T, n[i], k, k, k, n[i], 1, 1, 0, 0, ws, ws_bytes, st));
    return EZL_OK;
}

// dw_i[n_i, k] (=|+=) dy_i[T, n_i]^T x[T, k], the dy_i with a row stride of ld, into fp32 or bf16; a null target is skipped
int weight_gradients(int count, const void* const* dy, int64_t ld, const void* x, const ezl_layer_grad* g, int64_t T, const int64_t* n, int64_t k,
                     void* ws, int64_t ws_bytes, void* st) {
    void* out[3];
    int acc[3];
    const int64_t ks[3] = {k, k, k}, lds[3] = {ld, ld, ld};
    const void* xs[3] = {x, x, x};
    bool one = count > 1;
    for (int i = 0; i < count; ++i) {
        out[i] = g[i].f32 ? g[i].f32 : g[i].bf16;
        acc[i] = g[i].accumulate;
        one = one && out[i] && (g[i].f32 != nullptr) == (g[0].f32 != nullptr);
    }
    if (one && ezl_gemm_group_form_workspace_bytes(0, count, n, ks, T) >= 0)
        return ezl_gemm_bf16_group(count, dy, xs, out, n, ks, T, lds, ks, ks, 0, 0, g[0].f32 ? 1 : 0, acc, ws, ws_bytes, st);
    for (int i = 0; i < count; ++i)
        if (out[i])
            EZL_TRY(ezl_gemm_bf16(dy[i], x, out[i], n[i], k, T, ld, k, k, 0, 0, g[i].f32 ? 1 : 0, acc[i], ws, ws_bytes, st));
    return EZL_OK;
}

// gradient list entries of the weights, in WeightGradients' order
constexpr int kWeights[kGemmListMax] = {EZL_G_Q, EZL_G_K, EZL_G_V, EZL_G_O, EZL_G_GATE, EZL_G_UP, EZL_G_DOWN};

// all weight gradients in one launch: all wanted, in one type, and estimated to be faster than piece by piece
bool in_one_list(const Dims& m, const ezl_layer_grad* g) {
    for (int i : kWeights)
        if (!(g[i].f32 || g[i].bf16) || (g[i].f32 != nullptr) != (g[EZL_G_Q].f32 != nullptr)) return false;
    return WeightGradients(m).list_bytes(m.T, g[EZL_G_Q].f32 ? 4 : 2) >= 0;
}

// elements of the parameters, in the order of the gradient list
void parameter_sizes(const Dims& m, int64_t (&n)[EZL_G_COUNT]) {
    n[EZL_G_LN1] = n[EZL_G_LN2] = m.h;
    n[EZL_G_Q] = n[EZL_G_O] = m.qw * m.h;
    n[EZL_G_K] = n[EZL_G_V] = m.kw * m.h;
    n[EZL_G_GATE] = n[EZL_G_UP] = n[EZL_G_DOWN] = m.f * m.h;
    n[EZL_G_BQ] = m.qw;
    n[EZL_G_BK] = n[EZL_G_BV] = m.kw;
}
bool gradients_meet(const Dims& m, const ezl_layer_grad* g) {
    int64_t n[EZL_G_COUNT];
    parameter_sizes(m, n);
    const char *from[EZL_G_COUNT], *to[EZL_G_COUNT];
    for (int i = 0; i < EZL_G_COUNT; ++i) {
        from[i] = (const char*)(g[i].f32 ? g[i].f32 : g[i].bf16);
        to[i] = from[i] + (from[i] ? n[i] * (g[i].f32 ? 4 : 2) : 0);
        for (int j = 0; j < i; ++j)
            if (from[i] < to[j] && from[j] < to[i]) return true;
    }
    return false;
}

int check(const char* name, const ezl_layer* l) {
    EZL_REQUIRE(l, EZL_EINVAL, "%s: null argument", name);
    EZL_REQUIRE(l->s > 0 && l->b > 0 && l->h > 0 && l->nq > 0 && l->nk > 0 && l->nq % l->nk == 0 && l->d > 0 && l->f > 0 && l->ndocs > 0,
                EZL_EINVAL, "%s: bad sizes", name);
    EZL_REQUIRE((l->bq != nullptr) == (l->bk != nullptr) && (l->bq != nullptr) == (l->bv != nullptr), EZL_EINVAL,
                "%s: q, k and v biases go together", name);
    return EZL_OK;
}

}  // namespace

extern "C" int64_t ezl_layer_bytes(const ezl_layer* l, int which) {
    if (check("ezl_layer_bytes", l)) return -1;
    const Dims m(*l);
    if (which == 0) return Saved(m, nullptr).bytes;
    if (which == 1) return ForwardTemp(*l, m, nullptr).bytes;
    if (which == 2) return BackwardTemp(*l, m, nullptr).bytes;
    return -1;
}

extern "C" int ezl_layer_plan(const ezl_layer* l, int fp32) {
    if (check("ezl_layer_plan", l)) return -1;
    const Dims m(*l);
    return WeightGradients(m).list_bytes(m.T, fp32 ? 4 : 2) >= 0;
}

extern "C" int ezl_layer_fwd(const ezl_layer* l, const void* x, void* y, void* saved, void* temp, void* st) {
    EZL_TRY(check("ezl_layer_fwd", l));
    EZL_REQUIRE(x && y && saved && temp, EZL_EINVAL, "ezl_layer_fwd: null pointer");
    EZL_REQUIRE(ezl_aligned16(y), EZL_EINVAL, "ezl_layer_fwd: y must be 16-byte aligned");
    const Dims m(*l);
    const Saved a(m, saved);
    const ForwardTemp t(*l, m, temp);
    const int64_t row_q[2] = {l->b * m.qw, m.qw}, row_k[2] = {l->b * m.kw, m.kw};  // (sequence, batch) strides
    EZL_TRY(ezl_rmsnorm_fwd(x, nullptr, l->ln1, a.n1, nullptr, a.rstd1, m.T, m.h, l->eps1, st));
    {
        const void* w[3] = {l->wq, l->wk, l->wv};
        const int64_t n[3] = {m.qw, m.kw, m.kw};
        void* out[3] = {a.q, a.k, a.v};
        void* raw[3] = {t.bias_in, (char*)t.bias_in + m.T * m.qw * 2, (char*)t.bias_in + m.T * (m.qw + m.kw) * 2};
        EZL_TRY(forward_products(3, a.n1, w, l->bq ? raw : out, m.T, n, m.h, t.ws, t.ws_bytes, st));
        const void* bias[3] = {l->bq, l->bk, l->bv};
        if (l->bq)
            EZL_TRY(qkv_bias_rope(raw, bias, out, m.nq, m.nk, m.d, l->cos, l->sin, l->position_ids, l->s, l->b, l->npos, (hipStream_t)st));
        else
            EZL_TRY(ezl_rope_apply_pair(a.q, a.q, m.nq, m.qw, m.qw, a.k, a.k, m.nk, m.kw, m.kw, l->cos, l->sin, l->position_ids, l->s, l->b,
                                        m.d, l->npos, 0, st));
    }
    const int64_t b1 = l->b > 1;
    const int64_t strides[8] = {row_q[0], b1 * row_q[1], row_k[0], b1 * row_k[1], row_k[0], b1 * row_k[1], row_q[0], b1 * row_q[1]};
    EZL_TRY(ezl_attn_fwd(a.q, a.k, a.v, a.ctx, a.lse, l->cu_seqlens, l->ndocs, m.T, l->s, m.nq, m.nk, m.d, l->scale, strides, st));
    EZL_TRY(ezl_gemm_bf16(a.ctx, l->wo, t.wide, m.T, m.h, m.qw, m.qw, m.qw, m.h, 1, 1, 0, 0, t.ws, t.ws_bytes, st));
    // A small layer's result begins as the residual sum, to which the down projection adds its product in its epilogue: a launch that adds the two takes 4 us
    // there, nearly all of it the launch.  With more to add, the epilogue waits longer for the sum than that launch takes.  us of a layer, launch and epilogue: 1024 x 256
    // 209.4, 207.2; 2048 x 768 576, 573.4; 1531 x 4096 3020, 3027; 4000 x 2048 2662, 2675 (whole passes per layer): the lines cross between 1.6 and 6.3 million elements.
    const int64_t bytes = m.T * m.h * 2;
    const bool apart = (const char*)y + bytes <= (const char*)x || (const char*)x + bytes <= (const char*)y;  // (y is written before x is read for the last time)
    const bool sum_in_epilogue = apart && m.T * m.h <= 5 << 19;
    EZL_TRY(rmsnorm_fwd_keep_sum(t.wide, x, l->ln2, a.n2, a.sum, sum_in_epilogue ? y : nullptr, a.rstd2, m.T, m.h, l->eps2, st));
    {
        const void* w[2] = {l->wg, l->wu};
        const int64_t n[2] = {m.f, m.f};
        void* out[2] = {a.gate, a.up};
        EZL_TRY(forward_products(2, a.n2, w, out, m.T, n, m.h, t.ws, t.ws_bytes, st));
    }
    EZL_TRY(ezl_swiglu_fwd(a.gate, a.up, a.act, m.T * m.f, st));
    if (sum_in_epilogue) return gemm_forward_add(a.act, l->wd, y, m.T, m.h, m.f, t.ws, t.ws_bytes, st);
    EZL_TRY(ezl_gemm_bf16(a.act, l->wd, t.wide, m.T, m.h, m.f, m.f, m.f, m.h, 1, 1, 0, 0, t.ws, t.ws_bytes, st));
    return ezl_add(t.wide, a.sum, y, m.T * m.h, st);
}

extern "C" int ezl_layer_bwd(const ezl_layer* l, const void* x, const void* dy, void* dx, const void* saved, void* temp, const ezl_layer_grad* g,
                             void* st) {
    EZL_TRY(check("ezl_layer_bwd", l));
    EZL_REQUIRE(x && dy && dx && saved && temp && g, EZL_EINVAL, "ezl_layer_bwd: null pointer");
    const Dims m(*l);
    const Saved a(m, const_cast<void*>(saved));
    const BackwardTemp t(*l, m, temp);
    EZL_REQUIRE((g[EZL_G_LN1].f32 || g[EZL_G_LN1].bf16) && (g[EZL_G_LN2].f32 || g[EZL_G_LN2].bf16), EZL_EINVAL,
                "ezl_layer_bwd: the norm weights' gradients are part of their kernels");
    EZL_REQUIRE(!gradients_meet(m, g), EZL_EINVAL, "ezl_layer_bwd: two gradients share memory (they are written in the kernels' order)");
    const bool one_list = in_one_list(m, g);  // then their operands stay where they are to the end
    // y = sum + down(act): dy goes to both
    EZL_TRY(ezl_gemm_bf16(dy, l->wd, t.dact, m.T, m.f, m.h, m.h, m.f, m.f, 1, 0, 0, 0, t.ws, t.ws_bytes, st));
    if (!one_list) {
        const void* d[1] = {dy};
        EZL_TRY(weight_gradients(1, d, m.h, a.act, &g[EZL_G_DOWN], m.T, &m.h, m.f, t.ws, t.ws_bytes, st));
    }
    EZL_TRY(ezl_swiglu_bwd(t.dact, a.gate, a.up, t.dgate, t.dup, m.T * m.f, st));
    {
        const void *d[2] = {t.dgate, t.dup}, *w[2] = {l->wg, l->wu};
        const int64_t n[2] = {m.f, m.f};
        EZL_TRY(ezl_gemm_bf16_ksplit(2, d, w, t.dn, m.T, m.h, n, m.f, m.h, m.h, 1, 0, 0, 0, t.ws, t.ws_bytes, st));
        if (!one_list) EZL_TRY(weight_gradients(2, d, m.f, a.n2, &g[EZL_G_GATE], m.T, n, m.h, t.ws, t.ws_bytes, st));
    }
    NormWeightGrad ln1, ln2;
    EZL_TRY(rmsnorm_bwd_rows(t.dn, a.sum, l->ln2, a.rstd2, dy, t.dsum, g[EZL_G_LN2].f32 ? nullptr : g[EZL_G_LN2].bf16, g[EZL_G_LN2].f32,
                             g[EZL_G_LN2].accumulate, t.ln2_sums, m.T, m.h, ln2, st));
    // sum = x + o(ctx)
    EZL_TRY(ezl_gemm_bf16(t.dsum, l->wo, t.dctx, m.T, m.qw, m.h, m.h, m.qw, m.qw, 1, 0, 0, 0, t.ws, t.ws_bytes, st));
    if (!one_list) {
        const void* d[1] = {t.dsum};
        EZL_TRY(weight_gradients(1, d, m.h, a.ctx, &g[EZL_G_O], m.T, &m.h, m.qw, t.ws, t.ws_bytes, st));
    }
    const int64_t S = m.qw + 2 * m.kw;
    bf16_t *dq = (bf16_t*)t.dqkv, *dk = dq + m.qw, *dv = dk + m.kw;
    const int64_t b1 = l->b > 1, qs = l->b * m.qw, qb = b1 * m.qw, ks = l->b * m.kw, kb = b1 * m.kw, ds = l->b * S, db = b1 * S;
    const int64_t strides[16] = {qs, qb, ks, kb, ks, kb, qs, qb, qs, qb, ds, db, ds, db, ds, db};
    EZL_TRY(ezl_attn_bwd(a.q, a.k, a.v, a.ctx, t.dctx, a.lse, t.delta, dq, dk, dv, l->cu_seqlens, l->ndocs, m.T, l->s, m.nq, m.nk, m.d, l->scale,
                         strides, t.ws, t.ws_bytes, st));
    EZL_TRY(ezl_rope_apply_pair(dq, dq, m.nq, S, S, dk, dk, m.nk, S, S, l->cos, l->sin, l->position_ids, l->s, l->b, m.d, l->npos, 1, st));
    {
        const void *d[3] = {dq, dk, dv}, *w[3] = {l->wq, l->wk, l->wv};
        const int64_t n[3] = {m.qw, m.kw, m.kw};
        if (l->bq) {
            QkvBiasGrad gb;
            for (int i = 0; i < 3; ++i) {
                gb.f32[i] = (float*)g[EZL_G_BQ + i].f32;
                gb.bf16[i] = (bf16_t*)g[EZL_G_BQ + i].bf16;
                gb.accumulate[i] = g[EZL_G_BQ + i].accumulate;
            }
            EZL_TRY(qkv_bias_grad(t.dqkv, gb, m.T, m.qw, m.kw, t.ws, (hipStream_t)st));
        }
        EZL_TRY(ezl_gemm_bf16_ksplit(3, d, w, t.dn, m.T, m.h, n, S, m.h, m.h, 1, 0, 0, 0, t.ws, t.ws_bytes, st));
        if (!one_list) EZL_TRY(weight_gradients(3, d, S, a.n1, &g[EZL_G_Q], m.T, n, m.h, t.ws, t.ws_bytes, st));
    }
    if (one_list) {
        const WeightGradients w(m);
        const void *d[kGemmListMax] = {dq, dk, dv, t.dsum, t.dgate, t.dup, dy};
        const void *x[kGemmListMax] = {a.n1, a.n1, a.n1, a.ctx, a.n2, a.n2, a.act};
        const int64_t ld[kGemmListMax] = {S, S, S, m.h, m.f, m.f, m.h};
        void* out[kGemmListMax];
        int acc[kGemmListMax];
        for (int i = 0; i < kGemmListMax; ++i) {
            const ezl_layer_grad& target = g[kWeights[i]];
            out[i] = target.f32 ? target.f32 : target.bf16;
            acc[i] = target.accumulate;
        }
        EZL_TRY(gemm_list(kGemmListMax, d, x, out, w.n, w.k, m.T, ld, w.k, w.k, 0, 0, g[EZL_G_Q].f32 ? 1 : 0, acc, t.ws, t.ws_bytes, st));
    }
    EZL_TRY(rmsnorm_bwd_rows(t.dn, x, l->ln1, a.rstd1, t.dsum, dx, g[EZL_G_LN1].f32 ? nullptr : g[EZL_G_LN1].bf16, g[EZL_G_LN1].f32,
                             g[EZL_G_LN1].accumulate, t.ws, m.T, m.h, ln1, st));
    return norm_weight_grads(ln1, ln2, m.h, st);
}
