"""Kernels at the sizes where a launch rule or a tile edge can go wrong, against plain fp32 PyTorch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from easyllm_amd import kernels
    return kernels


def rnd(*shape, seed=0, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * scale).bfloat16()


@pytest.mark.parametrize("rows,h", [(1, 1032), (7, 1152), (515, 1280), (4099, 1536), (3, 1544)])
@pytest.mark.parametrize("fused", [False, True])
def test_rmsnorm_fwd_widths_that_do_not_divide_a_block(K, rows, h, fused):
    """192 threads per row (1024 < h <= 1536) do not divide a 256-thread block.  One fp32 result rounded to bf16: half an
    ulp (2^-9 of the value), plus fp32 sums of h terms in another order (far below)."""
    print("rmsnorm", rows, h, fused, flush=True)
    x, w = rnd(rows, h, seed=1), (1 + 0.1 * rnd(h, seed=2).float()).bfloat16()
    r = rnd(rows, h, seed=3) if fused else None
    y, rstd, s = K.rmsnorm_fwd(x, w, 1e-6, residual=r)
    z = (x.float() + r.float()).bfloat16() if fused else x
    if fused:
        assert torch.equal(s, z)
    ref_rstd = torch.rsqrt(z.float().square().mean(-1) + 1e-6)
    ref = z.float() * ref_rstd[:, None] * w.float()
    assert ((y.float() - ref).abs() <= ref.abs() * (2 ** -8) + 1e-6).all()
    assert torch.allclose(rstd, ref_rstd, rtol=1e-5)


# ---- GEMM ------------------------------------------------------------------------------------------------------------
def gemm_bound(A, B):
    """Per element: K products of bf16 values are exact in fp32; summing K of them in any order is off by at most
    K 2^-24 sum|a b| (taken 4 times too large); one rounding to bf16 on top where the result is bf16."""
    K = A.shape[1]
    return A.float().abs() @ B.float().abs() * (4 * K * 2.0 ** -24)


def check_gemm(K, form, M, N, Kd, accumulate=False, seed=0):
    """form 0 forward, 1 input gradient, 2 weight gradient with an fp32 result, 3 weight gradient with a bf16 result."""
    A = rnd(M, Kd, seed=seed) if form < 2 else rnd(Kd, M, seed=seed).t()
    B = rnd(N, Kd, seed=seed + 1).t() if form == 0 else rnd(Kd, N, seed=seed + 1)
    dt = torch.float32 if form == 2 else torch.bfloat16
    out = rnd(M, N, seed=seed + 2).to(dt) if accumulate else torch.full((M, N), float("nan"), device="cuda", dtype=dt)
    ref = A.float() @ B.float() + (out.float() if accumulate else 0)
    lda, ldb = max(A.stride()), max(B.stride())
    K.gemm(A if form < 2 else A.t(), B.t() if form == 0 else B, M, N, Kd, lda, ldb, form < 2, form == 0, out=out, accumulate=accumulate)
    tol = gemm_bound(A, B) + (ref.abs() * 2.0 ** -8 if dt == torch.bfloat16 else ref.abs() * 2.0 ** -22) + 1e-6
    worst = ((out.float() - ref).abs() - tol).max().item()
    assert worst <= 0, (form, M, N, Kd, accumulate, worst)


@pytest.mark.parametrize("form,M,N,Kd", [
    (0, 1024, 256, 688), (0, 300, 520, 8), (0, 256, 256, 56), (0, 256, 264, 4104), (1, 1024, 256, 688), (1, 257, 512, 72),
    (2, 688, 256, 1531), (2, 256, 4096, 1), (2, 264, 248, 4097), (2, 512, 512, 63), (3, 256, 264, 65)])
def test_gemm_k_tails(K, form, M, N, Kd):
    """Reductions that are no multiple of the 64-wide K tile: the last tile's missing k read as zero."""
    print("gemm", form, M, N, Kd, flush=True)
    check_gemm(K, form, M, N, Kd)
    check_gemm(K, form, M, N, Kd, accumulate=True, seed=5)


@pytest.mark.parametrize("T,n_in,outs", [(300, 256, (688, 688)), (1024, 256, (256, 64, 72)), (129, 520, (8, 1000, 120))])
def test_gemm_input_gradient_over_pairs_with_k_tails(K, T, n_in, outs):
    print("dgrad multi", T, n_in, outs, flush=True)
    ld = max(outs)
    dys = [torch.zeros(T, ld, device="cuda", dtype=torch.bfloat16)[:, :o].copy_(rnd(T, o, seed=i)) for i, o in enumerate(outs)]
    for dy, o in zip(dys, outs):  # what follows a row's valid part must not reach the result
        if o < ld:
            torch.as_strided(dy, (T, ld - o), (ld, 1), dy.storage_offset() + o).fill_(float("nan"))
    ws = [rnd(o, n_in, seed=10 + i) for i, o in enumerate(outs)]
    dx = K.linear_dgrad_multi(dys, ws)
    A, B = torch.cat([d.contiguous() for d in dys], 1), torch.cat(ws, 0)
    ref = A.float() @ B.float()
    assert ((dx.float() - ref).abs() <= gemm_bound(A, B) + ref.abs() * 2.0 ** -8 + 1e-6).all()


# (form, M, N, K) by the tile rows, columns and waves that a product of that size takes (test_call_forms.py holds the rule to this);
# forms: 0 forward, 1 input gradient, 2 weight gradient in fp32, 3 in bf16
SMALLER_TILES = {
    # the waves share the reduction: fewer and more K tiles than waves, a ragged tail, one row, one vector of columns
    (64, 64, 8): [(0, 65, 72, 1000), (2, 256, 264, 1531), (1, 1, 8, 520), (3, 8, 64, 449)],
    # one and several K tiles per stage ring
    (64, 64, 4): [(0, 64, 64, 64), (0, 1167, 1024, 1024), (2, 2048, 776, 2048), (3, 1544, 1032, 64)],
    # whole and split, one to four K tiles, tails, ragged edges
    (128, 128, 4): [(1, 1000, 2056, 200), (2, 2824, 1000, 1167), (0, 4100, 1800, 512), (2, 1024, 1032, 12000), (3, 1024, 1024, 9001), (0, 4096, 2048, 64),
                    (1, 4096, 2048, 128), (2, 4096, 2048, 192), (0, 4096, 2048, 200), (3, 2048, 2048, 4000)],
    (192, 128, 4): [(1, 1167, 2816, 1032), (1, 1531, 4096, 712)],
    (256, 128, 4): [(1, 700, 3080, 5128)],
    (256, 256, 8): [(0, 4001, 2056, 2048)]}
WIDE_TILES = {
    # K tails, ragged edges, element-wise stores, reductions split two to nine ways
    (192, 128, 4): [(0, 1780, 2328, 344), (1, 742, 2720, 904), (0, 1099, 3819, 368), (0, 1531, 4096, 4096), (0, 392, 4688, 2680), (1, 453, 2752, 3368),
                    (0, 556, 952, 5752), (2, 3456, 1336, 400), (2, 2224, 2168, 403), (3, 904, 4848, 467), (2, 904, 2488, 2160), (3, 384, 3240, 2765)],
    # bf16 weight gradients: several tiles per workgroup, K tails, a long reduction
    (256, 256, 4): [(3, 4872, 5128, 1040), (3, 5000, 6000, 1101), (3, 4096, 4096, 3205)],
    (256, 128, 4): [(0, 1195, 4816, 696), (1, 1209, 5008, 672), (0, 3872, 1648, 720), (0, 1009, 2808, 3040), (1, 423, 4704, 3568)]}
LARGEST_TILES = {
    # several tiles per workgroup: ragged edges, K tails, a split last round, one K tile more or less than where the rule changes; one workgroup
    # per tile: whole rounds and split ones, input gradients
    (256, 256, 4): [(0, 5000, 20000, 1096), (0, 4096, 8192, 1024), (0, 4000, 17000, 4096), (0, 4000, 17000, 4104), (2, 5000, 20008, 1100),
                    (2, 4096, 4352, 4160), (0, 4096, 4096, 8200), (2, 3000, 3080, 9000), (1, 4096, 4096, 10240), (1, 4100, 6152, 10248)],
    (256, 256, 8): [(2, 8192, 8192, 2048)],  # rows of B a multiple of 16 KiB apart
    (256, 128, 4): [(1, 4100, 5128, 10248)]}


def products(table):
    return [case for cases in table.values() for case in cases]


@pytest.mark.parametrize("form,M,N,Kd", products(SMALLER_TILES))
def test_gemm_smaller_tiles(K, form, M, N, Kd):
    print("gemm", form, M, N, Kd, flush=True)
    check_gemm(K, form, M, N, Kd)
    check_gemm(K, form, M, N, Kd, accumulate=True, seed=5)


@pytest.mark.parametrize("form,M,N,Kd", products(WIDE_TILES))
def test_gemm_wide_tiles(K, form, M, N, Kd):
    print("gemm", form, M, N, Kd, flush=True)
    check_gemm(K, form, M, N, Kd)
    check_gemm(K, form, M, N, Kd, accumulate=True, seed=5)
    if form == 0:
        x, w = rnd(M, Kd, seed=1), rnd(N, Kd, seed=2)
        f = K.linear_fwd(x, w, fp32_output=True)
        tol = gemm_bound(x, w.t()) + f.abs() * 2.0 ** -8 + 1e-6
        assert torch.equal(f, f.bfloat16().float()) and ((f - x.float() @ w.float().t()).abs() <= tol).all()


# (T, h, widths) of dx = sum of dy_i w_i by tile and waves
PAIRS = {(64, 64, 4): [(1167, 1024, (1024, 256, 256))], (64, 64, 8): [(1024, 256, (256, 256, 256))], (192, 128, 4): [(2048, 768, (2048, 2056))],
         (256, 128, 4): [(700, 3072, (3072, 1024, 1032)), (4000, 2048, (2048, 2048, 2056))]}
PAIRS_WIDE = {(192, 128, 4): [(742, 2720, (304, 304, 296)), (453, 2752, (1128, 1120, 1120))]}


@pytest.mark.parametrize("T,n_in,outs", products(PAIRS))
def test_gemm_input_gradient_over_pairs_on_smaller_tiles(K, T, n_in, outs):
    print("dgrad multi", T, n_in, outs, flush=True)
    ld = max(outs)
    dys = [torch.empty(T, ld, device="cuda", dtype=torch.bfloat16)[:, :o].copy_(rnd(T, o, seed=i)) for i, o in enumerate(outs)]
    ws = [rnd(o, n_in, seed=10 + i) for i, o in enumerate(outs)]
    A, B = torch.cat([d.contiguous() for d in dys], 1), torch.cat(ws, 0)
    ref = A.float() @ B.float()
    dx = K.linear_dgrad_multi(dys, ws)
    assert ((dx.float() - ref).abs() <= gemm_bound(A, B) + ref.abs() * 2.0 ** -8 + 1e-6).all()
    K.linear_dgrad_multi(dys, ws, out=dx, accumulate=True)
    assert ((dx.float() - 2 * ref).abs() <= 2 * gemm_bound(A, B) + ref.abs() * 2.0 ** -6 + 1e-6).all()


@pytest.mark.parametrize("T,n_in,outs", products(PAIRS_WIDE))
def test_gemm_input_gradient_over_pairs_on_wide_tiles(K, T, n_in, outs):
    test_gemm_input_gradient_over_pairs_on_smaller_tiles(K, T, n_in, outs)


def test_gemm_smaller_tiles_leave_what_is_outside_the_result_alone(K):
    """The stores past a tile's last row or column drop out: neighbours of a result that is a view stay as they were."""
    for form, M, N, Kd, extra in ((0, 65, 72, 1000, 16), (0, 1001, 1000, 1024, 16), (0, 4001, 2056, 256, 16), (2, 1000, 1000, 1100, 16),
                                  (0, 65, 71, 1000, 9), (0, 1001, 1003, 1024, 11), (0, 4001, 2049, 256, 13), (0, 700, 3075, 3072, 9)):
        dt = torch.float32 if form == 2 else torch.bfloat16  # (odd widths: element-wise stores)
        big = torch.full((M + 3, N + extra), 7.0, device="cuda", dtype=dt)
        A = rnd(M, Kd, seed=1) if form == 0 else rnd(Kd, M, seed=1)
        B = rnd(N, Kd, seed=2) if form == 0 else rnd(Kd, N, seed=2)
        K.gemm(A, B, M, N, Kd, A.stride(0), B.stride(0), form == 0, form == 0, out=big[1:M + 1, 8:N + 8])
        Af, Bf = (A, B.t()) if form == 0 else (A.t(), B)
        ref = Af.float() @ Bf.float()
        assert ((big[1:M + 1, 8:N + 8].float() - ref).abs() <= gemm_bound(Af, Bf) + ref.abs() * 2.0 ** -8 + 1e-6).all(), (form, M, N, Kd)
        border = big.clone()
        border[1:M + 1, 8:N + 8] = 7.0
        assert (border == 7.0).all(), (form, M, N, Kd)


@pytest.mark.parametrize("form,M,N,Kd", products(LARGEST_TILES))
def test_gemm_four_wave_kernel(K, form, M, N, Kd):
    print("gemm", form, M, N, Kd, flush=True)
    check_gemm(K, form, M, N, Kd)
    check_gemm(K, form, M, N, Kd, accumulate=True, seed=5)
    if form == 0:
        x, w = rnd(M, Kd, seed=1), rnd(N, Kd, seed=2)
        f = K.linear_fwd(x, w, fp32_output=True)
        tol = gemm_bound(x, w.t()) + f.abs() * 2.0 ** -8 + 1e-6
        assert torch.equal(f, f.bfloat16().float()) and ((f - x.float() @ w.float().t()).abs() <= tol).all()


def test_gemm_four_wave_kernel_over_pairs(K):
    T, n_in, outs = 4100, 4104, (16392, 16392)
    print("dgrad multi", T, n_in, outs, flush=True)
    dys = [rnd(T, o, seed=i) for i, o in enumerate(outs)]
    ws = [rnd(o, n_in, seed=10 + i) for i, o in enumerate(outs)]
    A, B = torch.cat(dys, 1), torch.cat(ws, 0)
    ref, bound = A.float() @ B.float(), gemm_bound(A, B)
    dx = K.linear_dgrad_multi(dys, ws)
    assert ((dx.float() - ref).abs() <= bound + ref.abs() * 2.0 ** -8 + 1e-6).all()
    K.linear_dgrad_multi(dys, ws, out=dx, accumulate=True)
    assert ((dx.float() - 2 * ref).abs() <= 2 * bound + ref.abs() * 2.0 ** -6 + 1e-6).all()


# split last rounds, K tails, ragged tiles, widths that differ: all in one launch of 256 x 256 tiles
FORWARD_LISTS = [(1726, 3072, (9920, 9920)), (1726, 3080, (9920, 9912)), (2050, 2056, (5504, 5504, 2056)), (4000, 2048, (5504, 5504))]


@pytest.mark.parametrize("T,n_in,outs", FORWARD_LISTS)
def test_gemm_forward_products_in_one_launch_on_the_largest_tiles(K, T, n_in, outs):
    print("gemm forward list", T, n_in, outs, flush=True)
    from easyllm_amd import _lib
    x, ws = rnd(T, n_in, seed=1), [rnd(o, n_in, seed=2 + i) for i, o in enumerate(outs)]
    assert _lib.gemm_group_form_workspace_bytes(True, (T,) * len(outs), outs, n_in) >= 0
    for y, w in zip(K.linear_fwd_multi(x, ws), ws):
        ref = x.float() @ w.float().t()
        assert ((y.float() - ref).abs() <= gemm_bound(x, w.t()) + ref.abs() * 2.0 ** -8 + 1e-6).all()


@pytest.mark.parametrize("T,n_in,outs", [(1024, 256, (256, 256, 256)), (1167, 1024, (1024, 256, 264)), (389, 768, (2048, 2056)),
                                         (17, 264, (8, 1000, 72)), (4000, 2048, (2048, 512, 512)), (9000, 256, (256, 512))])
def test_gemm_products_in_one_launch(K, T, n_in, outs):
    """q / k / v (gate / up) forward and weight gradients, all of sizes for which both share a launch, each against its own reference;
    and accumulation switched per product."""
    print("gemm group", T, n_in, outs, flush=True)
    from easyllm_amd import _lib
    x, ws = rnd(T, n_in, seed=1), [rnd(o, n_in, seed=2 + i) for i, o in enumerate(outs)]
    n = len(outs)
    assert _lib.gemm_group_form_workspace_bytes(True, (T,) * n, outs, n_in) >= 0
    assert _lib.gemm_group_form_workspace_bytes(False, outs, (n_in,) * n, T) >= 0
    for y, w in zip(K.linear_fwd_multi(x, ws), ws):
        ref = x.float() @ w.float().t()
        assert ((y.float() - ref).abs() <= gemm_bound(x, w.t()) + ref.abs() * 2.0 ** -8 + 1e-6).all()
    dys = [rnd(T, o, seed=7 + i) for i, o in enumerate(outs)]
    for dt in (torch.float32, None):
        accs = [i % 2 == 1 and dt is not None for i in range(n)]
        mgs = [None if dt is None else torch.full((o, n_in), 3.0, device="cuda", dtype=dt) for o in outs]
        for dw, dy, acc in zip(K.linear_wgrad_multi(dys, x, mgs, accs), dys, accs):
            ref = dy.float().t() @ x.float() + (3.0 if acc else 0.0)
            assert dw.dtype == (dt or torch.bfloat16)
            tol = gemm_bound(dy.t(), x) + ref.abs() * (2.0 ** -22 if dt else 2.0 ** -8) + 1e-6
            assert ((dw.float() - ref).abs() <= tol).all()


# (h, nq, nk, f, b, s, fp32) of a layer by the tile and waves of its seven weight gradients in one list; None: in pieces
LAYER_LISTS = {
    (64, 64, 4): [(64, 1, 1, 72, 1, 3, True)],
    (64, 64, 8): [(256, 4, 1, 688, 2, 511, True)],
    # one, two or several K tiles per wave, K tails, split reductions
    (128, 128, 4): [(768, 12, 12, 2048, 2, 1024, True), (256, 4, 4, 1000, 1, 16001, True)],
    (192, 128, 4): [(1024, 16, 4, 2816, 3, 389, False)],
    # a split last round, with a K tail, ragged tiles, less than a round, more results than the cache holds, bf16
    (256, 256, 4): [(1024, 8, 8, 2816, 1, 4000, True), (2048, 16, 16, 5504, 1, 2048, True), (2048, 16, 4, 5504, 2, 1001, True),
                    (1920, 15, 15, 5056, 1, 2503, True), (1024, 8, 2, 3328, 1, 4003, True), (2944, 23, 23, 8360, 1, 987, True),
                    (2048, 16, 4, 5504, 1, 2961, False), (1792, 14, 14, 4672, 1, 4608, False)],
    None: [(2944, 23, 23, 9216, 1, 1691, True)]}


@pytest.mark.parametrize("h,nq,nk,f,b,s,main_grads", products(LAYER_LISTS))
def test_weight_gradients_of_a_layer_in_one_launch(h, nq, nk, f, b, s, main_grads):
    """A layer's seven weight gradients as one list of tiles, overwritten and then added to, against the composed layer's separate products: activations and
    their gradients are the same bits, the sums over the tokens are in fp32 in another order (bf16 results: one rounding apart)."""
    from easyllm_amd import runner
    print("weight gradients of a layer", h, f, b, s, flush=True)
    results = []
    for flops in (1e13, 0.0):
        torch.manual_seed(5)
        model = runner.build_model({"type": "llama_custom", "kwargs": dict(
            num_layers=1, hidden_size=h, num_attention_heads=nq, num_kv_attention_heads=nk, intermediate_size=f, vocab_size=512, seq_length=s,
            bf16=True, checkpoint_activations=False)}).cuda()
        layer = next(m for m in model.modules() if hasattr(m, "native_call_flops"))
        layer.native_call_flops = flops
        if main_grads:
            runner.attach_main_grads(model)
        g = torch.Generator().manual_seed(1)
        tokens, labels = (torch.randint(0, 512, (b, s), generator=g).cuda() for _ in range(2))
        for _ in range(2 if main_grads else 1):  # the second pass adds
            runner.forward_step(model, (tokens, torch.arange(s).expand(b, s).contiguous().cuda(), None), (labels, torch.ones(b, s, device="cuda")))
        results.append({n: (p.main_grad if main_grads else p.grad.float()) for n, p in layer.named_parameters() if p.dim() == 2})
    got, want = results
    assert len(want) == 7
    for n in want:
        assert (got[n] - want[n]).norm() <= (1e-5 if main_grads else 2.0 ** -8) * want[n].norm(), n


def attention_reference(q, k, v, do, cu):
    """(out, lse, dq, dk, dv) in float64 on the GPU; documents cu over the (b s) tokens."""
    s, b, nq, d = q.shape
    nk, scale = k.shape[2], d ** -0.5
    Q, KK, V, DO = (x.transpose(0, 1).reshape(s * b, -1, d).transpose(0, 1).double().contiguous() for x in (q, k, v, do))
    out, dq, dk, dv = torch.zeros_like(Q), torch.zeros_like(Q), torch.zeros_like(KK), torch.zeros_like(V)
    lse = torch.zeros(nq, s * b, device=q.device, dtype=torch.float64)
    for a, e in zip(cu[:-1], cu[1:]):
        later = torch.ones(e - a, e - a, dtype=torch.bool, device=q.device).triu(1)
        for h in range(nq):
            g = h // (nq // nk)
            S = (Q[h, a:e] @ KK[g, a:e].t() * scale).masked_fill(later, float("-inf"))
            P, dP = S.softmax(-1), DO[h, a:e] @ V[g, a:e].t()
            lse[h, a:e] = S.logsumexp(-1)
            out[h, a:e] = P @ V[g, a:e]
            dS = P * (dP - (dP * P).sum(-1, keepdim=True)) * scale
            dq[h, a:e] = dS @ KK[g, a:e]
            dk[g, a:e] += dS.t() @ Q[h, a:e]
            dv[g, a:e] += P.t() @ DO[h, a:e]
    back = lambda x: x.transpose(0, 1).reshape(b, s, -1, d).transpose(0, 1)
    return back(out), lse, back(dq), back(dk), back(dv)


# (d, nq, nk, b, s, documents) by what forward and backward take: 0 workgroups of 128 rows, 1 the same with key groups / in one launch, 2 of 32 rows
ATTENTION = {
    # one tile, tile edges, waves without a tile, more tiles than waves, grouped queries, documents
    (0, 2): [(64, 2, 2, 1, 1, None), (64, 4, 1, 3, 31, None), (128, 2, 2, 2, 33, None), (128, 4, 2, 1, 330, [0, 96, 97, 330]),
             (64, 2, 2, 2, 128, [0, 100, 128, 200, 256])],
    (2, 2): [(64, 3, 3, 1, 255, None), (128, 2, 1, 1, 257, None), (64, 4, 4, 2, 512, None), (128, 3, 3, 1, 65, None), (64, 8, 8, 1, 97, None),
             (64, 4, 2, 1, 700, [0, 300, 700]), (128, 6, 6, 1, 900, [0, 1, 450, 900]), (64, 2, 1, 1, 2048, [0, 600, 601, 2048])],
    (2, 1): [(128, 3, 1, 1, 640, None), (64, 12, 4, 1, 1000, [0, 255, 1000]), (64, 16, 16, 1, 800, [0, 97, 800])],
    # the last tile missing for a key group, documents, split groups
    (1, 1): [(64, 24, 24, 2, 385, None), (128, 16, 4, 3, 449, None), (128, 24, 24, 1, 513, None), (64, 12, 12, 1, 2048, [0, 1, 66, 700, 2048]),
             (128, 8, 8, 1, 1030, [0, 64, 193, 1030])],
    (0, 1): [(64, 60, 60, 2, 100, None), (64, 8, 2, 1, 389, [0, 1, 2, 65, 129, 200, 389])],
    (1, 0): [(128, 38, 38, 1, 1025, None)],
    (0, 0): [(128, 30, 15, 4, 130, None), (64, 64, 64, 8, 140, None), (64, 40, 8, 1, 641, [0, 63, 64, 330, 641]), (128, 40, 40, 1, 700, [0, 129, 700])]}


@pytest.mark.parametrize("d,nq,nk,b,s,cu", products(ATTENTION))
def test_attention_for_every_split_of_the_work(K, d, nq, nk, b, s, cu):
    """Against float64.  Inputs are exact; probabilities, dS and the results are rounded to bf16 (2^-9 each): 1e-2 of a result's norm.
    dS is a difference that may cancel (a document of one token: exactly), off by scale |K| |dO . (O - its bf16 value)|."""
    print("attention", d, nq, nk, b, s, cu, flush=True)
    q, do = rnd(s, b, nq, d, seed=1), rnd(s, b, nq, d, seed=2)
    kv = rnd(s, b, 2 * nk + 1, d, seed=3)  # strides other than the heads' width
    k, v = kv[:, :, :nk], kv[:, :, nk:2 * nk]
    cut = None if cu is None else torch.tensor(cu, device="cuda", dtype=torch.int32)
    want = attention_reference(q, k, v, do, cu or [i * s for i in range(b + 1)])
    out, lse = K.attn_fwd(q, k, v, cut)
    got = (out, lse) + tuple(K.attn_bwd(q, k, v, out, do, lse, cut))
    assert (lse - want[1]).abs().max() <= 1e-4
    for name, x, w, cancels in zip(("out", "lse", "dq", "dk", "dv"), got, want, (0, 0, 1, 1, 0)):
        assert (x.double() - w).norm() <= 1e-2 * w.norm() + cancels * 2.0 ** -8 * do.double().norm(), name
    q[s // 2, 0, 0, 3] = float("nan")  # one query: its row of the result, nobody else's
    out2, _ = K.attn_fwd(q, k, v, cut)
    assert out2[s // 2, 0, 0].isnan().all()
    out2[s // 2, 0, 0] = out[s // 2, 0, 0]
    assert torch.equal(out2, out)


@pytest.mark.parametrize("nq,s,ndocs", [(512, 16, 33000), (128, 129, 70000)])
def test_attention_with_more_documents_than_one_axis_of_a_launch_holds(K, nq, s, ndocs):
    """All but the first document are empty.  Workgroups for all documents and heads on one axis would be 2^32 threads or more, which no launch
    takes.  Against the one document by itself: other kernels at these sizes, so 1e-2 of a result's norm as for every split of the work."""
    print("attention, empty documents", nq, s, ndocs, flush=True)
    q, k, v, do = (rnd(s, 1, n, 64, seed=i) for i, n in ((1, nq), (2, nq // 4), (3, nq // 4), (4, nq)))
    one = torch.tensor([0, s], device="cuda", dtype=torch.int32)
    many = torch.cat([one, torch.full((ndocs - 1,), s, device="cuda", dtype=torch.int32)])
    results = []
    for cu in (one, many):
        out, lse = K.attn_fwd(q, k, v, cu)
        results.append((out, lse) + tuple(K.attn_bwd(q, k, v, out, do, lse, cu)))
    for name, a, b in zip(("out", "lse", "dq", "dk", "dv"), *results):
        assert (a.double() - b.double()).norm() <= 1e-2 * a.double().norm(), name


def test_swiglu_results_larger_than_the_last_level_cache(K):
    """Written past the caches: the same bits as in four calls of a quarter of the size."""
    print("swiglu beyond the cache", flush=True)
    n = (140 << 20) + 32
    g, u, do = (rnd(n // 8, 8, seed=i) for i in (1, 2, 3))
    out, (dg, du) = K.swiglu_fwd(g, u), K.swiglu_bwd(do, g, u)
    for i in range(4):
        part = slice(i * n // 32, (i + 1) * n // 32)
        a, b = K.swiglu_bwd(do[part], g[part], u[part])
        assert torch.equal(out[part], K.swiglu_fwd(g[part], u[part])) and torch.equal(dg[part], a) and torch.equal(du[part], b)


@pytest.mark.parametrize("rows,h", [(270000, 520), (70001, 2048), (50000, 3080), (34608, 4096), (23001, 6144), (17500, 8192)])
def test_rmsnorm_backward_with_results_larger_than_the_last_level_cache(K, rows, h):
    """Written past the caches: the same bits as for its parts; the weight's gradient over all rows against float64 sums of the parts' (partial sums of
    up to rows / 256 products each in fp32: 1e-4)."""
    print("rmsnorm backward beyond the cache", rows, h, flush=True)
    x, dy, dr, w = rnd(rows, h, seed=1), rnd(rows, h, seed=2), rnd(rows, h, seed=3), rnd(h, seed=4)
    rstd = (x.float().square().mean(1) + 1e-5).rsqrt()
    mg = torch.empty(h, device="cuda")
    dx, _ = K.rmsnorm_bwd(dy, x, w, rstd, dresidual=dr, main_grad=mg)
    total = torch.zeros(h, device="cuda", dtype=torch.float64)
    for i in range(4):
        part, sub = slice(i * rows // 4, (i + 1) * rows // 4), torch.empty(h, device="cuda")
        assert torch.equal(dx[part], K.rmsnorm_bwd(dy[part], x[part], w, rstd[part], dresidual=dr[part], main_grad=sub)[0])
        total += sub.double()
    assert (mg.double() - total).norm() <= 1e-4 * total.norm()


@pytest.mark.parametrize("sizes", [[1], [4096, 4095, 4097, 3], [0, 8, 0, 70001], [1 + 37 * i for i in range(101)]])
def test_optimizer_over_lists_of_tensors(K, sizes):
    """Chunk edges, empty tensors and more tensors than one launch takes: the norm against fp64, the update bit for bit against
    the single-tensor call."""
    print("optimizer lists", len(sizes), flush=True)
    gs = [torch.randn(n, device="cuda") for n in sizes]
    partials = torch.full((K.sumsq_list_partials(len(sizes)),), float("nan"), device="cuda")
    K.sumsq_list(gs, partials)
    want = sum(g.double().square().sum().item() for g in gs)
    assert abs(partials.double().sum().item() - want) <= 1e-5 * want
    coef = torch.tensor([5.0, 0.5], device="cuda")
    one = [[torch.randn(n, device="cuda") for n in sizes] for _ in range(2)] + [[torch.rand(n, device="cuda") for n in sizes]]
    lst = [[t.clone() for t in ts] for ts in one]
    params = [torch.zeros(n, device="cuda", dtype=torch.bfloat16) if i % 3 else None for i, n in enumerate(sizes)]
    params1 = [None if p is None else p.clone() for p in params]
    K.adamw_list(*lst, gs, params, 1e-2, 0.9, 0.95, 1e-8, 0.1, 3, True, coef)
    for i in range(len(sizes)):
        K.adamw_step(one[0][i], one[1][i], one[2][i], gs[i], params1[i], 1e-2, 0.9, 0.95, 1e-8, 0.1, 3, True, coef)
        assert all(torch.equal(a[i], b[i]) for a, b in zip(one, lst))
        if params[i] is not None:
            assert torch.equal(params[i], params1[i]) and torch.equal(params[i], lst[0][i].bfloat16())


@pytest.mark.parametrize("name", ["mha", "gqa", "bias", "bf16_grads", "packed", "frozen", "checkpoint"])
def test_layer_in_one_native_call_equals_the_composed_layer(name):
    """Same kernels in the same order: loss and every gradient bit for bit, except where the composed form rounds once more
    (unequal q / kv widths: the input gradients of q, k and v are added in bf16 instead of in fp32)."""
    from easyllm_amd import data, runner
    h, nq = 256, 4
    nk = 1 if name in ("gqa", "packed") else 4
    kw = dict(num_layers=2, hidden_size=h, num_attention_heads=nq, num_kv_attention_heads=nk, intermediate_size=688, vocab_size=512,
              seq_length=192, bf16=True, checkpoint_activations=name == "checkpoint")
    if name == "bias":
        kw["transformer_layer_params"] = {"attention_qkv_bias": True}
    b, s = (1, 384) if name == "packed" else (2, 192)
    tokens = torch.randint(0, 512, (b, s), generator=torch.Generator().manual_seed(1)).cuda()
    labels = torch.randint(0, 512, (b, s), generator=torch.Generator().manual_seed(2)).cuda()
    pos = torch.arange(s).expand(b, s).contiguous().cuda()
    inputs = (tokens, pos, None)
    if name == "packed":
        cu = [0, 100, 101, 384]
        inputs = (tokens, torch.tensor([data.get_position_ids(cu)]).cuda(), None, torch.tensor(cu).cuda())
    results = []
    for flops in (1e12, 0.0):
        torch.manual_seed(3)
        model = runner.build_model({"type": "llama_custom", "kwargs": dict(kw)}).cuda()
        for m in model.modules():
            if hasattr(m, "native_call_flops"):
                m.native_call_flops = flops
        with torch.no_grad():
            for p in model.parameters():
                if p.dim() == 1:
                    p.add_(0.1 * torch.randn_like(p))
        if name == "frozen":
            for n, p in model.named_parameters():
                p.requires_grad_("q_proj" in n or "layernorm" in n or "up_proj" in n)
        if name != "bf16_grads":
            runner.attach_main_grads(model)
        nodes = []
        out = model(inputs)
        fn = out.grad_fn
        while fn is not None:
            nodes.append(type(fn).__name__)
            fn = fn.next_functions[0][0] if fn.next_functions else None
        if name != "checkpoint":
            assert any("DecoderLayer" in n for n in nodes) == (flops > 0)
        for _ in range(2):  # the second pass adds to the gradients
            loss = runner.forward_step(model, inputs, (labels, torch.ones(b, s, device="cuda")))
        grads = {n: (p.main_grad if hasattr(p, "main_grad") else p.grad) for n, p in model.named_parameters() if p.requires_grad}
        results.append((out.float(), loss, {n: g.float() for n, g in grads.items()}))
    (out1, loss1, g1), (out0, loss0, g0) = results
    assert torch.equal(out1, out0) and torch.equal(loss1, loss0) and g1.keys() == g0.keys()
    for n in g0:
        if nk == nq:
            assert torch.equal(g1[n], g0[n]), n
        else:  # 2 roundings of 2^-9 each in one layer's input gradient, carried through the layers below
            assert (g1[n] - g0[n]).norm() <= 2e-2 * g0[n].norm(), n


def test_a_hooked_submodule_keeps_the_composed_layer():
    from easyllm_amd import runner
    model = runner.build_model({"type": "llama_custom", "kwargs": dict(num_layers=1, hidden_size=128, num_attention_heads=2, intermediate_size=256,
                                                                       vocab_size=512, seq_length=64, bf16=True)}).cuda()
    seen = []
    model.get_submodule("3").mlp.register_forward_hook(lambda m, i, o: seen.append(o[0].shape))
    tokens = torch.randint(0, 512, (1, 64)).cuda()
    model((tokens, torch.arange(64).view(1, 64).cuda(), None))
    assert seen == [torch.Size([64, 1, 128])]


def test_hooks_on_biased_projections_and_on_the_head_run():
    """They see what the modules return by themselves: q with its bias, logits in bf16."""
    from easyllm_amd import runner
    model = runner.build_model({"type": "llama_custom", "kwargs": dict(
        num_layers=1, hidden_size=128, num_attention_heads=2, intermediate_size=256, vocab_size=512, seq_length=64, bf16=True,
        transformer_layer_params={"attention_qkv_bias": True})}).cuda()
    head = model.get_submodule("6")
    seen = {}
    tokens = torch.randint(0, 512, (1, 64)).cuda()
    inputs = (tokens, torch.arange(64).view(1, 64).cuda(), None)
    plain = model(inputs)
    hooks = [model.get_submodule("3").self_attn.q_proj.register_forward_hook(lambda m, i, o: seen.update(q=o[0].shape)),
             head.register_forward_hook(lambda m, i, o: seen.update(logits=o))]
    hooked = model(inputs)
    assert seen["q"] == torch.Size([64, 1, 128]) and seen["logits"].dtype == torch.bfloat16
    assert plain.dtype == hooked.dtype == torch.float32 and torch.equal(hooked, seen["logits"].float()) and torch.equal(hooked, plain)
    for hook in hooks:
        hook.remove()
    assert head(rnd(1, 64, 128)).dtype == torch.bfloat16


def test_gradient_buffers_of_another_size_are_refused():
    from easyllm_amd import runner
    model = runner.build_model({"type": "llama_custom", "kwargs": dict(num_layers=1, hidden_size=128, num_attention_heads=2, intermediate_size=256,
                                                                       vocab_size=512, seq_length=64, bf16=True,
                                                                       checkpoint_activations=False)}).cuda()
    tokens = torch.randint(0, 512, (1, 64)).cuda()
    out = model((tokens, torch.arange(64).view(1, 64).cuda(), None))
    runner.attach_main_grads(model)
    model.get_submodule("3").mlp.up_proj.weight.main_grad = torch.zeros(255, 128, device="cuda")
    with pytest.raises(ValueError, match="gradient buffer"):
        out.sum().backward()


@pytest.mark.parametrize("M,N,Kd", [(1024, 256, 256), (1167, 50304, 1024), (300, 1003, 72), (4096, 4096, 3136), (64, 72, 2000), (700, 3072, 3072)])
def test_gemm_forward_with_an_fp32_result_of_bf16_values(K, M, N, Kd):
    """Bit for bit the cast of the bf16 result: at one size both forms take the same tiles and the same split of the reduction, and
    every kernel adds the K tiles of a share in order."""
    print("gemm rounded fp32", M, N, Kd, flush=True)
    x, w = rnd(M, Kd, seed=1), rnd(N, Kd, seed=2)
    y, f = K.linear_fwd(x, w), K.linear_fwd(x, w, fp32_output=True)
    assert f.dtype == torch.float32 and torch.equal(f, f.bfloat16().float())
    assert torch.equal(f, y.float())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,V,cut", [(1, 8, 0), (37, 1000, 0), (5, 16384 + 8, 3), (300, 32000, 0), (9, 152064, 1000), (3, 2048, 2047)])
def test_loss_without_gradient_equals_the_fused_loss(K, rows, V, cut, dtype):
    """Same sums in another order: 1e-6 relative; ignored rows contribute exactly nothing, whatever they hold."""
    print("ce loss", rows, V, cut, dtype, flush=True)
    logits = (torch.randn(rows, V, device="cuda") * 4).to(dtype)
    labels = torch.randint(0, V, (rows,), device="cuda")  # (some fall into the cut columns: masked)
    weights = (torch.rand(rows, device="cuda") < 0.8).float()
    weights[0] = 1.0
    logits[weights == 0] = float("nan")
    count = weights.sum().view(1)
    want, _ = K.ce_fused(logits.clone(), labels, weights, count, cut, inplace=True)
    got = K.ce_loss(logits, labels, weights, cut)
    assert torch.allclose(got, want, rtol=1e-6, atol=2e-6)
    assert (got[weights == 0] == 0).all()


def test_default_fp32_logits_are_the_cast_of_the_bf16_ones():
    from easyllm_amd import runner
    kw = dict(num_layers=1, hidden_size=256, num_attention_heads=4, intermediate_size=512, vocab_size=1000, seq_length=64, bf16=True)
    tokens, pos = torch.randint(0, 1000, (2, 64)).cuda(), torch.arange(64).expand(2, 64).contiguous().cuda()
    target = (tokens, torch.ones(2, 64, device="cuda"))
    outs = []
    for fp32 in (True, False):
        torch.manual_seed(0)
        model = runner.build_model({"type": "llama_custom", "kwargs": dict(kw, fp32_logits=fp32)}).cuda()
        with torch.no_grad():
            no_grad_loss = model.loss_fn(model((tokens, pos, None)), target)
        out = model((tokens, pos, None))
        loss = model.loss_fn(out, target)
        loss.backward()
        assert abs(no_grad_loss.item() - loss.item()) <= 1e-6 * loss.item()
        outs.append((out, {n: p.grad for n, p in model.named_parameters()}))
    assert outs[0][0].dtype == torch.float32 and torch.equal(outs[0][0], outs[1][0].float())
    for n in outs[0][1]:  # the logits' gradient is rounded to bf16 once either way, from exponentials of two kernels
        assert (outs[0][1][n].float() - outs[1][1][n].float()).norm() <= 2e-2 * outs[1][1][n].float().norm(), n


@pytest.mark.parametrize("ignored", [0.0, 0.3])
def test_a_training_step_needs_no_fp32_copy_of_the_logits(ignored):
    """forward_step with the default fp32 logits against its own composition: the same values in, fp32 inside, one rounding of the
    logits' gradient.  The two loss kernels add in another order: 1e-6 of the loss, and values of the rounded gradient that fall to the
    other side; the 12 bf16 tensors between it and the lowest weight gradient may each do so by one step, 2^-8 of a value, at
    most, independently of each other: sqrt(12) 2^-8."""
    from easyllm_amd import runner
    kw = dict(num_layers=1, hidden_size=256, num_attention_heads=4, intermediate_size=512, vocab_size=1000, seq_length=64, bf16=True)
    tokens, pos = torch.randint(0, 1000, (2, 64)).cuda(), torch.arange(64).expand(2, 64).contiguous().cuda()
    labels = torch.randint(0, 1000, (2, 64)).cuda()
    labels[torch.rand(2, 64, device="cuda") < ignored] = -100
    target = (labels, torch.ones(2, 64, device="cuda"))
    results = []
    for composed in (True, False):
        torch.manual_seed(0)
        model = runner.build_model({"type": "llama_custom", "kwargs": dict(kw)}).cuda()
        seen = []
        if composed:  # a hook on the model sees fp32 logits, as before
            model.register_forward_hook(lambda m, i, o: seen.append(o.dtype))
        loss = runner.forward_step(model, (tokens, pos, None), target)
        assert seen == [torch.float32] * composed
        results.append((loss, {n: p.grad.float() for n, p in model.named_parameters()}))
    (loss0, g0), (loss1, g1) = results
    assert abs(loss0.item() - loss1.item()) <= 1e-6 * loss0.item()
    for n in g0:
        assert (g0[n] - g1[n]).norm() <= 12 ** 0.5 * 2.0 ** -8 * g0[n].norm(), n


@pytest.mark.parametrize("V,h,rows,frequent", [(1, 8, 1, 0), (50, 64, 600, 0), (4099, 1024, 1167, 0), (4099, 1032, 1167, 700), (700, 4104, 130, 40),
                                               (90, 8200, 300, 100), (70000, 8192, 257, 33), (333, 512, 0, 0)])
def test_embedding_gradient_in_bf16_is_the_fp32_one_rounded(K, V, h, rows, frequent):
    """Every register depth of the kernel, frequent ids (more than 32 rows), a table of more than 1 GiB (cleared by a fill of its
    own) and an empty batch.  The sums run in fp32 in row order in both forms: equal bit for bit."""
    print("embedding gradient bf16", V, h, rows, frequent, flush=True)
    ids = torch.randint(0, V, (rows,), generator=torch.Generator().manual_seed(rows + h))
    ids[:frequent] = V // 2
    ids, dy = ids.cuda(), rnd(rows, h, seed=4)
    ref = torch.full((V, h), 3.5, device="cuda")
    K.embed_scatter_add(ids, dy, ref, accumulate=False)
    got = K.embed_grad_bf16(ids, dy, V)
    assert got.dtype is torch.bfloat16 and torch.equal(got, ref.bfloat16())


@pytest.mark.parametrize("V,h,rows,ids", [(32000, 256, 1024, "random"), (5000, 64, 4096, "distinct"), (50304, 72, 1167, "padding"), (131072, 64, 4095, "far apart"),
                                          (40, 128, 3000, "few"), (1, 8, 33, "random"), (131073, 64, 900, "random"), (300, 64, 500, "out of range"),
                                          # the largest of one workgroup, runs of equal ids, and between them ids out of range
                                          (5000, 64, 2048, "distinct"), (131072, 64, 1536, "far apart"), (3000, 72, 2047, "padding"),
                                          (40, 64, 1537, "few"), (700, 64, 1530, "runs"), (700, 64, 2049, "runs")])
def test_embedding_gradient_with_and_without_the_one_workgroup_tables(K, V, h, rows, ids):
    """Batches of up to 2048 rows (1536 where the buffer is overwritten) build their tables in one workgroup.  Rows with an id outside the table are skipped, so the same
    batch with 4097 of them behind it goes the general way: equal bit for bit, overwriting and adding."""
    print("embedding tables", V, h, rows, ids, flush=True)
    g = torch.Generator().manual_seed(rows)
    t = torch.randint(0, V, (rows,), generator=g)
    if ids == "distinct":
        t = torch.randperm(V, generator=g)[:rows]
    elif ids == "padding":
        t[rows // 2:] = 0
    elif ids == "far apart":
        t = torch.arange(rows) * 32 % V
    elif ids == "runs":
        t = torch.arange(rows) // 100 * 37 % V
        t[::9], t[5::64] = V, 3
    elif ids == "out of range":
        t[::7], t[::11] = V, -1
    long = torch.cat([t, torch.full((4097,), V)]).cuda()
    dy = torch.cat([rnd(rows, h, seed=4), torch.full((4097, h), float("nan"), device="cuda", dtype=torch.bfloat16)])
    for accumulate in (False, True):
        got, want = torch.full((V, h), 2.5, device="cuda"), torch.full((V, h), 2.5, device="cuda")
        K.embed_scatter_add(t.cuda(), dy[:rows].contiguous(), got, accumulate=accumulate)
        K.embed_scatter_add(long, dy, want, accumulate=accumulate)
        assert torch.equal(got, want)
    assert torch.equal(K.embed_grad_bf16(t.cuda(), dy[:rows].contiguous(), V), K.embed_grad_bf16(long, dy, V))


@pytest.mark.parametrize("rows,V,cut", [(3, 32776, 0), (700, 40960, 0), (2100, 40968, 0), (5, 50304, 304), (1167, 53256, 0), (9, 65536, 9), (4, 65544, 0),
                                        (6, 73720, 1000),
                                        # little more than a vector left, less than one, a whole number of them, all but the last column
                                        (3, 40960, 40951), (4, 50304, 50299), (3, 36872, 4104), (520, 65536, 1)])
def test_loss_and_gradient_of_rows_kept_as_bf16_in_registers(K, rows, V, cut):
    """Edges of the register counts, cut columns, ignored rows, labels in the cut, more rows than blocks; against float64.  The sum of V
    fp32 exponentials is off by V 2^-24 at most, the gradient by that and one rounding to bf16."""
    print("loss", rows, V, cut, flush=True)
    x = rnd(rows, V, seed=3, scale=2.0)
    labels = torch.randint(0, V - cut, (rows,), generator=torch.Generator().manual_seed(1)).cuda()
    labels[::5] = -100
    if cut:
        labels[1] = V - 1
    w, count = K.ce_prepare(labels, None, -100)
    loss, grad = K.ce_fused(x, labels, w, count, cut, inplace=False)
    for r in list(range(min(rows, 12))) + [rows - 1]:
        xd, t = x[r].double(), labels[r].item()
        if t == -100:
            assert loss[r] == 0 and (grad[r] == 0).all()
            continue
        masked = t >= V - cut
        lse = xd[:V - cut].logsumexp(0)
        want = lse - (xd[:V - cut].max() if masked else xd[t])
        assert abs(loss[r].double() - want) <= V * 2.0 ** -24 + 1e-5
        g = (xd - lse).exp()
        if not masked:
            g[t] -= 1
        g /= count.double()
        assert ((grad[r].double() - g).abs() <= g.abs() * (2.0 ** -8 + V * 2.0 ** -23) + 2.0 ** -126).all()
    assert torch.equal(K.ce_fused(x, labels, w, count, cut)[1], grad)  # in place: the same bits


@pytest.mark.parametrize("d0,d1,h", [(2, 3, 8), (2, 512, 256), (3, 389, 1024), (5, 7, 1032), (1000, 4, 2048), (2, 33, 2056), (3, 301, 4096), (7, 5, 5120), (2, 129, 8192)])
def test_rmsnorm_of_rows_in_the_other_order(K, d0, d1, h):
    """x [d0, d1, h] stored as [d1, d0, h]: what the norm of its contiguous copy gives, forward and backward, bit for bit."""
    print("rmsnorm swapped", d0, d1, h, flush=True)
    x, w, dy = rnd(d1, d0, h, seed=1).transpose(0, 1), rnd(h, seed=2), rnd(d0, d1, h, seed=3)
    assert K.rows_swapped(x)
    y, rstd = K.rmsnorm_fwd_swapped(x, w, 1e-6)
    want_y, want_rstd, _ = K.rmsnorm_fwd(x.contiguous(), w, 1e-6)
    assert y.is_contiguous() and torch.equal(y, want_y) and torch.equal(rstd, want_rstd)
    dx, dw = K.rmsnorm_bwd_swapped(dy, x, w, rstd)
    want_dx, want_dw = K.rmsnorm_bwd(dy, x.contiguous(), w, rstd)
    assert K.rows_swapped(dx) and torch.equal(dx, want_dx) and torch.equal(dw, want_dw)
    mg, want_mg = torch.full((h,), 0.5, device="cuda"), torch.full((h,), 0.5, device="cuda")
    K.rmsnorm_bwd_swapped(dy, x, w, rstd, main_grad=mg, accumulate=True)
    K.rmsnorm_bwd(dy, x.contiguous(), w, rstd, main_grad=want_mg, accumulate=True)
    assert torch.equal(mg, want_mg)


@pytest.mark.parametrize("d0,d1,h,V,same", [(2, 3, 8, 5, 0), (2, 512, 256, 32000, 0), (3, 389, 1024, 4099, 40), (4, 1000, 72, 900, 1500), (700, 3, 4104, 130, 300),
                                            (2, 257, 8200, 64, 33), (2, 33000, 8, 50, 65999)])
def test_embedding_of_rows_in_the_other_order(K, d0, d1, h, V, same):
    """ids [d0, d1], rows stored as [d1, d0, h]: the gather, its flags and every form of the gradient as of contiguous rows, bit for bit.  Ids that occur once,
    a few times, and (`same` of them) often enough for the kernel's lists and its bitmap over two windows of row numbers."""
    print("embedding swapped", d0, d1, h, V, same, flush=True)
    ids = torch.randint(0, V, (d0 * d1,), generator=torch.Generator().manual_seed(d0 + d1))
    ids[d0 * d1 - same:] = V // 2
    ids[0], ids[-1] = V, -1  # out of range
    ids, W, dy = ids.view(d0, d1).cuda(), rnd(V, h, seed=1), rnd(d1, d0, h, seed=2).transpose(0, 1)
    out, flag = K.embed_gather(ids, W, swapped=True)
    want, want_flag = K.embed_gather(ids, W)
    assert K.rows_swapped(out) and torch.equal(out, want) and flag.item() == want_flag.item() == 3
    host = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    out, none = K.embed_gather(ids, W, host, swapped=True)
    torch.cuda.synchronize()
    assert none is None and torch.equal(out, want) and host.item() == 0x101
    for accumulate in (False, True):
        got, ref = torch.full((V, h), 2.5, device="cuda"), torch.full((V, h), 2.5, device="cuda")
        assert K.embed_grad_swapped(ids, dy, V, got, accumulate) is None
        K.embed_scatter_add(ids, dy.contiguous(), ref, accumulate=accumulate)
        assert torch.equal(got, ref)
    assert torch.equal(K.embed_grad_swapped(ids, dy, V), K.embed_grad_bf16(ids, dy.contiguous(), V))


# (s, b, h, f) by the down projection's (tile rows, columns, split or not, waves); beyond 2.6 million elements a launch adds the two
RESIDUAL_SUMS = {
    (64, 64, False, 4): [(111, 1, 144, 128)],
    (64, 64, False, 8): [(46, 2, 80, 464), (192, 2, 256, 688)],
    (64, 64, True, 4): [(35, 1, 192, 1720)],
    (128, 128, False, 4): [(130, 2, 6912, 72)],
    (128, 128, True, 4): [(65, 1, 4192, 6016)],
    (192, 128, False, 4): [(1897, 3, 448, 640)],
    (192, 128, True, 4): [(2431, 1, 72, 11392)],
    (256, 128, True, 4): [(213, 1, 4208, 4056)],
    (192, 256, True, 4): [(143, 1, 1280, 28800)],
    (256, 256, True, 4): [(449, 1, 5632, 6016)],
    None: [(1280, 2, 1024, 1024), (1281, 2, 1024, 1024), (40, 1, 8200, 256), (301, 1, 8192, 512), (130, 3, 264, 8192)]}  # (and norms of every kind)


@pytest.mark.parametrize("want,case", [(w, c) for w, cs in RESIDUAL_SUMS.items() for c in cs])
def test_the_residual_sum_in_the_down_projections_epilogue(want, case):
    """The bits of the product, rounded, and an addition, from what the layer saved; a contiguous x of which y shares nothing stays as it was."""
    from easyllm_amd import _lib
    from easyllm_amd import functional as F_
    from easyllm_amd import kernels as K_
    s, b, h, f = case
    print("residual sum", want, case, flush=True)
    _, rows, cols, split, waves = _lib.gemm_plan("forward", [s * b], [h], f)
    assert want is None or (rows, cols, split > 1, waves) == want
    heads, d, T = 2, 64, s * b
    sizes = [(h,), (heads * d, h), (heads * d, h), (heads * d, h), (h, heads * d), (h,), (f, h), (f, h), (h, f)]
    ws = [rnd(*n, seed=i, scale=0.05 if len(n) > 1 else 1.0) for i, n in enumerate(sizes)]
    x = rnd(s, b, h, seed=20)
    before, angles = x.clone(), torch.rand(s, d // 2, device="cuda")
    cos, sin = angles.cos(), angles.sin()  # (they have to outlive the call)
    y, saved = K_.layer_fwd(K_.layer_desc(x.shape, (heads, heads, d), f, (1e-5, 1e-5), d ** -0.5, ws, None, cos, sin, None, None), x)
    at, parts = 0, {}  # the saved block: pieces on 256 bytes each
    for name, count, size in (("n1", T * h, 2), ("rstd1", T, 4), ("q", T * heads * d, 2), ("k", T * heads * d, 2), ("v", T * heads * d, 2), ("ctx", T * heads * d, 2),
                              ("lse", heads * T, 4), ("sum", T * h, 2), ("n2", T * h, 2), ("rstd2", T, 4), ("gate", T * f, 2), ("up", T * f, 2), ("act", T * f, 2)):
        parts[name] = saved[at:at + count * size].view(torch.bfloat16 if size == 2 else torch.float32)
        at += (count * size + 255) // 256 * 256
    assert at == saved.numel()
    o = K_.linear_fwd(parts["ctx"].view(T, heads * d), ws[4])
    assert torch.equal(F_.add(o, x.view(T, h)), parts["sum"].view(T, h))
    assert torch.equal(K_.swiglu_fwd(parts["gate"], parts["up"]), parts["act"])
    assert torch.equal(y.view(T, h), F_.add(K_.linear_fwd(parts["act"].view(T, f), ws[8]), parts["sum"].view(T, h)))
    assert torch.equal(x, before)
