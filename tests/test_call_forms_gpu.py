"""Forms of calls that a fast path must answer as the general one does: shared and odd buffers, replaced parts, values that are not
finite."""
import ctypes

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


def product_bound(A, B):
    """Products of bf16 values are exact in fp32; summing K of them in any order is off by at most K 2^-24 sum|a b| (taken 4 times
    too large)."""
    return A.float().abs() @ B.float().abs() * (4 * A.shape[1] * 2.0 ** -24)


def small_model(**kw):
    from easyllm_amd import runner
    torch.manual_seed(3)
    cfg = dict(num_layers=1, hidden_size=256, num_attention_heads=4, intermediate_size=688, vocab_size=512, seq_length=192, bf16=True,
               checkpoint_activations=False)
    cfg.update(kw)
    model = runner.build_model({"type": "llama_custom", "kwargs": cfg}).cuda()
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn_like(p))
    return model


def small_batch(b=2, s=192, vocab=512):
    g = torch.Generator().manual_seed(1)
    tokens, labels = torch.randint(0, vocab, (b, s), generator=g).cuda(), torch.randint(0, vocab, (b, s), generator=g).cuda()
    return (tokens, torch.arange(s).expand(b, s).contiguous().cuda(), None), (labels, torch.ones(b, s, device="cuda"))


def decoder_layer(model):
    return next(m for m in model.modules() if hasattr(m, "native_call_flops"))


# ---- results of one launch that share memory ---------------------------------------------------------------------------
@pytest.mark.parametrize("T,n_in,n_out,count", [(1024, 256, 256, 3), (1167, 1024, 256, 2), (4000, 2048, 512, 3), (9000, 256, 512, 2)])
def test_weight_gradients_of_one_weight_used_several_times(K, T, n_in, n_out, count):
    """One buffer for several products, at sizes where they would otherwise share a launch: they are added one after the other."""
    from easyllm_amd import _lib
    print("one weight, several uses", T, n_in, n_out, count, flush=True)
    assert _lib.gemm_group_form_workspace_bytes(False, (n_out,) * count, (n_in,) * count, T) >= 0
    x, dys = rnd(T, n_in, seed=1), [rnd(T, n_out, seed=2 + i) for i in range(count)]
    total = sum(dys[i].double().t() @ x.double() for i in range(count))
    bound = sum(product_bound(dy.t(), x) for dy in dys) + total.abs() * 2.0 ** -20 + 1e-5
    for first in (False, True):
        mg = torch.full((n_out, n_in), 3.0, device="cuda")
        K.linear_wgrad_multi(dys, x, [mg] * count, [first] + [True] * (count - 1))
        assert ((mg - (total + 3.0 * first)).abs() <= bound).all()


def test_a_weight_shared_by_two_projections_through_autograd():
    from easyllm_amd import functional as F_
    T, n = 1024, 256
    x = rnd(T, n, seed=1)
    w = torch.nn.Parameter(rnd(n, n, seed=2))
    w.main_grad, w.main_grad_fresh = torch.full((n, n), 7.0, device="cuda"), True
    dys = [rnd(T, n, seed=3 + i) for i in range(2)]
    torch.autograd.backward(F_.fan_out_linear(x, w, w), dys)
    ref = sum(dy.double().t() @ x.double() for dy in dys)
    bound = sum(product_bound(dy.t(), x) for dy in dys) + ref.abs() * 2.0 ** -20 + 1e-5
    assert ((w.main_grad - ref).abs() <= bound).all() and not w.main_grad_fresh


def test_weight_gradients_into_buffers_with_far_apart_rows(K):
    """Rows 8 MiB apart are more than the smaller-tile kernels' offsets reach: such results are stored by the others."""
    from easyllm_amd import _lib
    T, n_in, outs, ld = 1024, 264, (8, 16), 1 << 21
    assert _lib.gemm_group_form_workspace_bytes(False, outs, (n_in,) * 2, T) >= 0
    x, dys = rnd(T, n_in, seed=1), [rnd(T, o, seed=2 + i) for i, o in enumerate(outs)]
    bufs = [torch.full((o * ld,), 5.0, device="cuda") for o in outs]
    mgs = [b.as_strided((o, n_in), (ld, 1)) for b, o in zip(bufs, outs)]
    K.linear_wgrad_multi(dys, x, mgs, [False, True])
    for mg, buf, dy, old in zip(mgs, bufs, dys, (0.0, 5.0)):
        ref = dy.double().t() @ x.double() + old
        assert ((mg - ref).abs() <= product_bound(dy.t(), x) + ref.abs() * 2.0 ** -20 + 1e-5).all()
        mg.fill_(5.0)
        assert (buf == 5.0).all()


@pytest.mark.parametrize("tied", ["norms", "k_v", "gate_up", "q_o", "biases"])
@pytest.mark.parametrize("fresh", [True, False])
def test_a_layer_with_a_shared_parameter_against_the_composed_layer(tied, fresh):
    """The same activations and gradients of activations bit for bit; the weight gradients from the same bf16 values, summed in
    fp32 in another order at most: 1e-5 of their norm."""
    from easyllm_amd import runner
    print("shared parameter", tied, fresh, flush=True)
    results = []
    for flops in (1e12, 0.0):
        model = small_model(num_layers=2, **({"transformer_layer_params": {"attention_qkv_bias": True}} if tied == "biases" else {}))
        for m in model.modules():
            if hasattr(m, "native_call_flops"):
                m.native_call_flops = flops
                attn, mlp = m.self_attn, m.mlp
                if tied == "norms":
                    m.post_attention_layernorm.weight = m.input_layernorm.weight
                elif tied == "k_v":
                    attn.v_proj.weight = attn.k_proj.weight
                elif tied == "gate_up":
                    mlp.up_proj.weight = mlp.gate_proj.weight
                elif tied == "q_o":
                    attn.o_proj.weight = attn.q_proj.weight
                else:
                    attn.v_proj.bias = attn.k_proj.bias = attn.q_proj.bias
        runner.attach_main_grads(model)
        for p in model.parameters():
            p.main_grad.fill_(3.0)
            p.main_grad_fresh = fresh
        loss = runner.forward_step(model, *small_batch())
        results.append((loss, {n: p.main_grad for n, p in model.named_parameters()}))
    (loss1, g1), (loss0, g0) = results
    assert torch.equal(loss1, loss0) and g1.keys() == g0.keys()
    for n in g0:
        assert (g1[n] - g0[n]).norm() <= 1e-5 * g0[n].norm(), n


# ---- optimizer lists ---------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("order", [(0, 1, 0), (0, 0, 0, 0), tuple(range(50)) + (3, 49, 3), (1,) * 60])
def test_a_tensor_that_occurs_twice_in_an_optimizer_list_is_updated_twice(K, order):
    """One after the other, as single-tensor calls in the order of the list: bit for bit."""
    print("optimizer list with repetitions", len(order), flush=True)
    sizes = [70001 if i == 0 else 4096 * (1 + i % 3) + i for i in range(max(order) + 1)]
    sides = []
    for _ in range(2):
        torch.manual_seed(5)
        sides.append([[torch.randn(n, device="cuda") for n in sizes], [torch.randn(n, device="cuda") for n in sizes],
                      [torch.rand(n, device="cuda") for n in sizes], [torch.randn(n, device="cuda") for n in sizes],
                      [torch.zeros(n, device="cuda", dtype=torch.bfloat16) for n in sizes]])
    coef = torch.tensor([5.0, 0.5], device="cuda")
    a, b = sides
    K.adamw_list(*[[ts[i] for i in order] for ts in a], 1e-2, 0.9, 0.95, 1e-8, 0.1, 3, True, coef)
    for i in order:
        K.adamw_step(*[ts[i] for ts in b], 1e-2, 0.9, 0.95, 1e-8, 0.1, 3, True, coef)
    assert all(torch.equal(x, y) for xs, ys in zip(a, b) for x, y in zip(xs, ys))


def test_the_gradient_norm_after_parameters_were_taken_out_of_a_group():
    """Fewer tensors than the optimizer was built with, over the edge of what one launch takes."""
    from easyllm_amd import optimizer
    params = []
    for i in range(50):
        p = torch.nn.Parameter(rnd(100 + i, seed=i))
        p.main_grad = torch.randn(100 + i, device="cuda")
        params.append(p)
    opt = optimizer.FusedAdam([{"params": params}])
    opt.global_grad_norm(1.0)
    for keep in (50, 48, 3):
        del opt.param_groups[0]["params"][keep:]
        want = torch.stack([p.main_grad.double().square().sum() for p in params[:keep]]).sum().sqrt()
        assert abs(opt.global_grad_norm(1.0)[0] - want) <= 1e-5 * want


def test_optimizer_lists_of_different_lengths_are_refused(K):
    lists = [[torch.zeros(8, device="cuda") for _ in range(2)] for _ in range(4)] + [[None, None]]
    for short in range(5):
        args = [ts[:1] if i == short else ts for i, ts in enumerate(lists)]
        with pytest.raises(ValueError, match="one entry per tensor"):
            K.adamw_list(*args, 1e-2, 0.9, 0.95, 1e-8, 0.1, 3)


# ---- loss without gradient ---------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V,cut", [(8, 0), (1000, 0), (4096, 8), (32000, 0), (16392, 3)])
def test_loss_without_gradient_on_values_that_are_not_finite(K, V, cut, dtype):
    """Row by row what the loss with gradient gives, NaN for NaN; -inf in a counted column is a probability of zero."""
    print("ce loss, not finite", V, cut, dtype, flush=True)
    nan, inf = float("nan"), float("inf")
    rows = 10
    logits = (torch.randn(rows, V, device="cuda", generator=torch.Generator(device="cuda").manual_seed(V)) * 4).to(dtype)
    labels = torch.full((rows,), V - cut - 1, device="cuda")
    logits[0, :8] = nan           # one vector of one thread, and nothing else of that thread if the row is short
    logits[1] = nan
    logits[2] = nan
    labels[2] = V                 # (a label outside the vocabulary)
    logits[3, V - cut - 1] = nan  # a single column, the last one
    logits[4, :V // 2] = -inf     # finite
    logits[5] = -inf
    logits[6] = -inf
    labels[6] = -1
    logits[7, 0] = inf
    logits[8, :8] = -inf
    logits[8, 7] = nan
    if V - cut - 1 > 8:
        logits[9, 1:V - cut - 1] = -inf  # finite
    if cut:
        logits[9, V - cut:] = nan        # (columns that are cut off are not looked at)
    weights = torch.ones(rows, device="cuda")
    want, _ = K.ce_fused(logits.clone(), labels, weights, weights.sum().view(1), cut, inplace=True)
    got = K.ce_loss(logits, labels, weights, cut)
    print(got.tolist(), want.tolist(), flush=True)
    assert torch.allclose(got, want, rtol=1e-6, atol=2e-6, equal_nan=True)
    assert got[[0, 1, 2, 3, 8]].isnan().all()


# ---- parts of a layer that a native call must not pass by --------------------------------------------------------------
def test_attention_dropout_is_refused_in_training():
    model, (inputs, _) = small_model(), small_batch()
    core = decoder_layer(model).self_attn.core_attention_flash
    core.dropout_p = 0.1
    with pytest.raises(NotImplementedError, match="dropout"):
        model(inputs)
    out = model.eval()(inputs)
    core.dropout_p = 0.0
    assert torch.equal(out, model(inputs))


@pytest.mark.parametrize("part,method", [("input_layernorm", "forward_keep_input"), ("post_attention_layernorm", "forward_with_residual"),
                                         ("self_attn.core_attention_flash", "forward_sb"), ("self_attn.rotary_emb", "tables"),
                                         ("self_attn", "forward"), ("mlp", "forward"), ("mlp.down_proj", "forward")])
@pytest.mark.parametrize("on_class", [False, True])
def test_a_replaced_method_of_a_submodule_is_called(monkeypatch, part, method, on_class):
    model, (inputs, _) = small_model(), small_batch()
    want = model(inputs)
    module = decoder_layer(model).get_submodule(part)
    calls = []
    original = getattr(type(module), method)
    if on_class:
        def replaced(self, *a, **kw):
            calls.append(method)
            return original(self, *a, **kw)
        monkeypatch.setattr(type(module), method, replaced)
    else:
        def replaced(*a, **kw):
            calls.append(method)
            return original(module, *a, **kw)
        monkeypatch.setattr(module, method, replaced)
    assert torch.equal(model(inputs), want) and calls


def test_forward_mode_through_the_fused_loss_is_refused():
    """Also where no reverse-mode gradient is wanted: a tangent must not be dropped without a word."""
    import torch.autograd.forward_ad as fwAD
    from easyllm_amd import functional as F_
    logits, labels = rnd(4, 64), torch.arange(4, device="cuda")
    with fwAD.dual_level():
        dual = fwAD.make_dual(logits, rnd(4, 64, seed=1))
        with pytest.raises(RuntimeError, match="(?i)forward"):
            F_.fused_cross_entropy_loss(dual, labels)


def test_a_loss_of_which_only_the_mask_wants_a_gradient():
    from easyllm_amd import functional as F_
    mask = torch.ones(4, device="cuda", requires_grad=True)
    logits, labels = rnd(4, 64), torch.arange(4, device="cuda")
    loss = F_.fused_cross_entropy_loss(logits, labels, mask)
    loss.backward()  # (the mask is not differentiated)
    assert mask.grad is None
    ref = torch.nn.functional.cross_entropy(logits.float(), labels)
    assert abs(loss.item() - ref.item()) <= 1e-5 * ref.item()


@pytest.mark.parametrize("without", [("k_proj",), ("k_proj", "v_proj")])
@pytest.mark.parametrize("flops", [1e12, 0.0])
def test_projections_of_which_some_have_no_bias(without, flops):
    """As with biases of zero there (the sum with a zero bias is exact)."""
    results = []
    for removed in (True, False):
        model, batch = small_model(transformer_layer_params={"attention_qkv_bias": True}), small_batch()
        layer = decoder_layer(model)
        layer.native_call_flops = flops
        for name in without:
            proj = layer.self_attn.get_submodule(name)
            if removed:
                proj.bias = None
            else:
                with torch.no_grad():
                    proj.bias.zero_()
        out = model(batch[0])
        loss = model.loss_fn(out, batch[1])
        loss.backward()
        results.append((out, loss, {n: p.grad.float() for n, p in model.named_parameters()}))
    (out1, loss1, g1), (out0, loss0, g0) = results
    assert torch.equal(out1, out0) and torch.equal(loss1, loss0) and set(g0) - set(g1) == {n for n in g0 if n.split(".")[-2] in without and n.endswith("bias")}
    for n in g1:  # (the input gradient of three separate projections is added in bf16: a rounding or two)
        assert (g1[n] - g0[n]).norm() <= 2e-2 * g0[n].norm(), n


def test_a_projection_that_leaves_its_bias_to_the_caller():
    """skip_bias_add: the projection's bias is not added by it, and the attention drops what it returns beside its result."""
    model, (inputs, _) = small_model(transformer_layer_params={"attention_qkv_bias": True}), small_batch()
    k = decoder_layer(model).self_attn.k_proj
    k.skip_bias_add = True
    out = model(inputs)
    k.skip_bias_add = False
    with torch.no_grad():
        k.bias.zero_()
    assert torch.equal(out, model(inputs))


def test_a_down_projection_with_a_bias_of_its_own():
    model, (inputs, _) = small_model(), small_batch()
    down = decoder_layer(model).mlp.down_proj
    down.bias, down.skip_bias_add = torch.nn.Parameter(rnd(256, seed=5)), False
    out = model(inputs)
    decoder_layer(model).native_call_flops = 0.0
    assert torch.equal(out, model(inputs))
    down.bias = None
    assert not torch.equal(out, model(inputs))


# ---- C entries ---------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("flag", [1, 2, -1, 3])
@pytest.mark.parametrize("entry,T,n_in,outs", [("ksplit", 1024, 256, (256, 64)), ("ksplit", 4096, 5120, (4096, 1024)), ("ksplit", 300, 264, (256,)),
                                               ("group", 1024, 256, (256, 64)), ("group", 9000, 256, (256, 512)), ("single", 1024, 256, (256,))])
def test_any_nonzero_accumulate_flag_adds(K, entry, T, n_in, outs, flag):
    from easyllm_amd import _lib
    print("accumulate", entry, T, n_in, outs, flag, flush=True)
    n = len(outs)
    vp, i64 = ctypes.c_void_p * n, ctypes.c_int64 * n
    ptr = lambda ts: vp(*[t.data_ptr() for t in ts])
    ld = max(outs)
    dys = [torch.empty(T, ld, device="cuda", dtype=torch.bfloat16)[:, :o].copy_(rnd(T, o, seed=i)) for i, o in enumerate(outs)]
    ws = torch.empty(64 << 20, device="cuda", dtype=torch.uint8)
    if entry == "ksplit":
        weights = [rnd(o, n_in, seed=9 + i) for i, o in enumerate(outs)]
        out = [torch.full((T, n_in), 3.0, device="cuda", dtype=torch.bfloat16)]
        _lib.call("ezl_gemm_bf16_ksplit", n, ptr(dys), ptr(weights), out[0].data_ptr(), T, n_in, i64(*outs), ld, n_in, n_in, 1, 0, 0, flag,
                  ws.data_ptr(), ws.numel(), None)
        torch.cuda.synchronize()
        ref = [3.0 + sum(dy.float() @ w.float() for dy, w in zip(dys, weights))]
        bound = [sum(product_bound(dy, w) for dy, w in zip(dys, weights)) + ref[0].abs() * 2.0 ** -8 + 1e-5]
    else:
        x = rnd(T, n_in, seed=9)
        out = [torch.full((o, n_in), 3.0, device="cuda") for o in outs]
        if entry == "group":
            _lib.call("ezl_gemm_bf16_group", n, ptr(dys), vp(*[x.data_ptr()] * n), ptr(out), i64(*outs), i64(*[n_in] * n), T, i64(*[ld] * n),
                      i64(*[n_in] * n), i64(*[n_in] * n), 0, 0, 1, (ctypes.c_int * n)(*[flag] * n), ws.data_ptr(), ws.numel(), None)
        else:
            _lib.call("ezl_gemm_bf16", dys[0].data_ptr(), x.data_ptr(), out[0].data_ptr(), outs[0], n_in, T, ld, n_in, n_in, 0, 0, 1, flag,
                      ws.data_ptr(), ws.numel(), None)
        torch.cuda.synchronize()
        ref = [3.0 + dy.float().t() @ x.float() for dy in dys]
        bound = [product_bound(dy.t(), x) + r.abs() * 2.0 ** -20 + 1e-5 for dy, r in zip(dys, ref)]
    for o, r, tol in zip(out, ref, bound):
        assert ((o.float() - r).abs() <= tol).all()


# ---- embedding gradient ------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("T,K_,outs", [(1024, 256, (256, 256, 256)), (17, 264, (8, 1000, 72)), (389, 2056, (768, 264)), (300, 5000, (128, 64))])
def test_input_gradients_in_one_launch(K, T, K_, outs):
    """The form of the group call that no wrapper uses: dy_i[T, K] w_i[K, n_i] in bf16, accumulation per product."""
    print("gemm group input gradients", T, K_, outs, flush=True)
    from easyllm_amd import _lib
    n = len(outs)
    nbytes = _lib.gemm_group_workspace_bytes((T,) * n, outs, K_)
    assert nbytes >= 0
    dys, ws = [rnd(T, K_, seed=i) for i in range(n)], [rnd(K_, o, seed=10 + i) for i, o in enumerate(outs)]
    dxs = [torch.full((T, o), 3.0, device="cuda", dtype=torch.bfloat16) for o in outs]
    accs = [i % 2 for i in range(n)]
    K.gemm_group(dys, ws, (T,) * n, outs, K_, [K_] * n, outs, True, False, dxs, accs, nbytes)
    for dx, dy, w, acc in zip(dxs, dys, ws, accs):
        ref = dy.float() @ w.float() + 3.0 * acc
        assert ((dx.float() - ref).abs() <= product_bound(dy, w) + ref.abs() * 2.0 ** -8 + 1e-6).all()


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("V,h,rows,counts", [
    (500, 64, 5000, (33, 256, 257, 1024, 1025, 2000)),      # ids on both sides of every limit of the ordering
    (40, 520, 9000, (2048, 2049, 3000, 40)),                # more rows of one id than the ordered list holds
    (300, 8, 140000, (33, 300, 2048, 65536, 60000)),        # several bitmap windows, full and nearly empty ones
    (3, 16, 65537, (65536,)), (2, 8, 131072, (131071, 1))])
def test_embedding_gradient_with_frequent_ids(K, V, h, rows, counts, accumulate):
    """Against the same sums taken in row order one row at a time (fp32, in the given order: bit for bit)."""
    print("embedding gradient, frequent ids", V, h, rows, counts, accumulate, flush=True)
    g = torch.Generator().manual_seed(rows)
    ids = torch.randint(len(counts), max(V, len(counts) + 1), (rows,), generator=g)
    where = torch.randperm(rows, generator=g)
    at = 0
    for i, n in enumerate(counts):
        ids[where[at:at + n]] = i
        at += n
    dy = torch.randn(rows, h, generator=g).bfloat16()
    old = torch.randn(V, h, generator=g)
    ref = torch.zeros(V, h)
    for i in ids.unique().tolist():
        ref[i] = torch.from_numpy(dy[ids == i].float().numpy().cumsum(axis=0, dtype="float32")[-1])
    out = old.cuda()
    K.embed_scatter_add(ids.cuda(), dy.cuda(), out, accumulate=accumulate)
    assert torch.equal(out.cpu(), ref + old if accumulate else ref)
    if not accumulate:
        assert torch.equal(K.embed_grad_bf16(ids.cuda(), dy.cuda(), V).cpu(), ref.bfloat16())


@pytest.mark.parametrize("s,b,h,f", [(512, 2, 256, 688), (389, 3, 1024, 2816), (389, 1, 768, 2048)])
def test_plans_of_a_repeated_step_are_not_searched_for_again(gpu_device, s, b, h, f):
    """A layer in one native call, forward and backward, which sizes its products' workspaces and launches them in turn: the second time nothing is searched for."""
    from easyllm_amd import _lib
    from easyllm_amd import functional as F_
    print("searches", s, b, h, f, flush=True)
    heads, d = h // 64, 64
    sizes = [(h,), (h, h), (h, h), (h, h), (h, h), (h,), (f, h), (f, h), (h, f)]
    ws = [rnd(*n, seed=i, scale=0.05 if len(n) > 1 else 1.0).requires_grad_(True) for i, n in enumerate(sizes)]
    x, angles = rnd(s, b, h, seed=20).requires_grad_(True), torch.rand(s, d // 2, device=gpu_device)

    def step():
        before = _lib.load().ezl_gemm_searches()
        y = F_.decoder_layer(x, ((heads, heads, d), f, (1e-5, 1e-5), d ** -0.5), angles.cos(), angles.sin(), None, None, tuple(ws))
        grads = torch.autograd.grad(y, [x] + ws, y.detach())
        assert all(torch.isfinite(g).all() for g in grads)
        return _lib.load().ezl_gemm_searches() - before

    with torch.autograd.set_multithreading_enabled(False):  # (a thread remembers its own)
        assert step() > 0
        assert step() == 0 and step() == 0
