"""Forms of calls that a fast path must answer as the general one does, where that can be seen without a GPU."""
import ctypes
import time

import pytest
import torch

import test_kernel_edges_gpu as edges
from easyllm_amd import _lib
from easyllm_amd import functional as F_


# the order in which a layer's backward writes its parameters' gradients (down, gate, up, ln2, o, q / k / v biases, q, k, v, ln1)
_WRITE_ORDER = (8, 6, 7, 5, 4, 9, 10, 11, 1, 2, 3, 0)


def _layer_with_fake_kernels(monkeypatch, params):
    """decoder_layer whose backward writes i + 1 as the gradient of parameter i, in the kernels' order and all reads of old values
    of a launch before its writes (the q / k / v and gate / up gradients are one launch each)."""
    def bwd(desc, x, dy, saved, targets):
        for launch in ((8,), (6, 7), (5,), (4,), (9, 10, 11), (1, 2, 3), (0,)):
            new = []
            for i in launch:
                if i < len(targets) and targets[i] is not None:
                    f32, bf16, acc = targets[i]
                    out = bf16 if f32 is None else f32
                    new.append((out, out + (i + 1) if acc else torch.full_like(out, i + 1)))
            for out, value in new:
                out.copy_(value)
        return torch.ones_like(x)

    monkeypatch.setattr(F_.K, "layer_desc", lambda *a: None)
    monkeypatch.setattr(F_.K, "layer_fwd", lambda desc, x: (x.clone(), torch.empty(0)))
    monkeypatch.setattr(F_.K, "layer_bwd", bwd)
    x = torch.ones(2, 1, 4, requires_grad=True)
    return F_.decoder_layer(x, (), torch.ones(1), torch.ones(1), None, None, tuple(params))


@pytest.mark.parametrize("fresh", [True, False])
@pytest.mark.parametrize("tied", [(0, 5), (1, 2), (2, 3), (6, 7), (10, 11), (1, 4), (0, 5, 1), (6, 7, 8)])
def test_a_parameter_that_occurs_twice_in_a_layer_gets_both_gradients(monkeypatch, tied, fresh):
    assert sorted(_WRITE_ORDER) == list(range(12))
    params = [torch.nn.Parameter(torch.zeros(4)) for _ in range(12)]
    for i in tied[1:]:
        params[i] = params[tied[0]]
    for p in params:
        p.main_grad = torch.full((4,), 100.0)
        p.main_grad_fresh = fresh
    _layer_with_fake_kernels(monkeypatch, params).sum().backward()
    for p in set(params):
        want = sum(i + 1 for i in range(12) if params[i] is p) + (0 if fresh else 100)
        assert torch.equal(p.main_grad, torch.full((4,), float(want))) and p.grad is None and not p.main_grad_fresh


def test_a_parameter_that_occurs_twice_in_a_layer_without_gradient_buffers(monkeypatch):
    params = [torch.nn.Parameter(torch.zeros(4)) for _ in range(9)]
    params[5], params[3] = params[0], params[2]
    _layer_with_fake_kernels(monkeypatch, params).sum().backward()
    assert params[0].grad[0] == 1 + 6 and params[2].grad[0] == 3 + 4 and params[1].grad[0] == 2


def test_layer_gradients_that_share_memory_are_refused():
    """The kernels write in their own order, several results in one launch; nothing is launched for such a call."""
    _lib.load()
    layer = _lib.Layer(s=8, b=1, h=64, nq=1, nk=1, d=64, f=64, ndocs=1, npos=8)
    grads = (_lib.LayerGrad * 12)()
    for i in range(9):
        grads[i].f32 = 0x100000 * (i + 1)
    grads[3].f32 = grads[2].f32 + 64 * 64 * 4 - 4  # v starts on the last element of k
    with pytest.raises(RuntimeError, match="share memory"):
        _lib.call("ezl_layer_bwd", ctypes.byref(layer), 256, 256, 256, 256, 256, grads, None)


def test_a_module_with_replaced_parts_is_not_plain(monkeypatch):
    from easyllm_amd import layers, transformer
    linear = lambda: layers.ColumnParallelLinear(8, 8, bias=False, use_cpu_initialization=True, params_dtype=torch.bfloat16)
    plain = lambda m, cls=layers.ColumnParallelLinear: transformer.is_plain(m, cls)
    norm = layers.RMSNorm(False, 8)
    assert plain(linear()) and plain(norm, layers.RMSNorm) and not plain(norm)
    for name in ("forward", "_call_impl", "_compiled_call_impl"):
        m = linear()
        m.__dict__[name] = m.forward
        assert not plain(m)
    for name in ("forward_keep_input", "forward_with_residual"):
        replaced = layers.RMSNorm(False, 8)
        replaced.__dict__[name] = norm.forward
        assert not plain(replaced, layers.RMSNorm)
    m = linear()
    handle = m.register_forward_hook(lambda *a: None)
    assert not plain(m)
    handle.remove()
    assert plain(m)
    monkeypatch.setattr(layers.ColumnParallelLinear, "forward", lambda self, x: (x, None))
    assert not plain(m) and plain(norm, layers.RMSNorm)


def test_a_replaced_loss_sees_the_logits_that_the_model_returns(monkeypatch):
    from easyllm_amd import losses, runner
    model = runner.build_model({"type": "llama_custom", "kwargs": dict(num_layers=1, hidden_size=64, num_attention_heads=1, intermediate_size=64,
                                                                       vocab_size=64, seq_length=8, bf16=True)})
    assert runner._logits_stay_inside(model)
    monkeypatch.setattr(losses.CrossEntropy, "__call__", lambda self, output, labels: output.sum())
    assert not runner._logits_stay_inside(model)


# (measured, us, as taken and, where both were, apart: forward; weight gradients)
@pytest.mark.parametrize("T,h,outs,forward,weight_gradient", [
    (1024, 256, (256, 256, 256), True, True),        # 5.8, 12.0; 8.1, 20.0
    (3072, 2048, (2048, 2048, 2048), True, True),    # 91, 89; 90, 132
    (2048, 4096, (4096, 1024, 1024), True, True),    # 91, 124; 115, 129
    (4096, 5120, (5120, 5120, 5120), True, False),   # 464, 548; apart
    (4096, 4096, (4096, 4096, 4096), False, False),
    (6144, 2048, (5504, 5504), True, True),          # 223, 238; 264, 264
    (1378, 4608, (12288, 12288), True, True),        # 276, 323; 434, 442
    (3600, 3072, (3072, 3072, 3072), True, True),    # 172, 188; 209, 269
    (1531, 4096, (11008, 11008), True, False),       # 208, 226; apart
    (8192, 5120, (13696, 13696), False, False)])
def test_products_of_256_tiles_share_a_launch_only_by_a_margin(T, h, outs, forward, weight_gradient):
    """The decision that linear_fwd_multi, linear_wgrad_multi and the whole-layer calls take."""
    n = len(outs)
    fwd, wgrad = ((T,) * n, outs, h), (outs, (h,) * n, T)
    assert (_lib.gemm_group_form_workspace_bytes(True, *fwd) >= 0) == forward
    assert (_lib.gemm_group_form_workspace_bytes(False, *wgrad) >= 0) == weight_gradient
    for sizes in (fwd, wgrad):  # a caller that does not say the form: one of the two decisions, and room for both
        forms = [_lib.gemm_group_form_workspace_bytes(a_kc, *sizes) for a_kc in (True, False)]
        assert _lib.gemm_group_workspace_bytes(*sizes) == (max(forms) if forms[0 if sizes[1][0] == sizes[2] else 1] >= 0 else -1)


# (measured, us: one launch of 128 rows against workgroups of 32)
@pytest.mark.parametrize("d,nq,nk,b,s,plan", [
    (64, 8, 1, 2, 500, 1),     # 23.2, 54.7
    (128, 4, 1, 2, 802, 1),    # 47.5, 67.5
    (128, 32, 4, 1, 79, 1),    # 17.1, 21.2
    (64, 2, 1, 3, 561, 2),     # 21.8, 19.4
    (64, 28, 7, 1, 83, 2),     # (three rows: 13.5, 11.2)
    (64, 4, 4, 2, 512, 2)])
def test_attention_backward_of_grouped_queries_on_32_rows_only_with_short_chains(d, nq, nk, b, s, plan):
    assert _lib.attn_plan(True, None, b * s, s, nq, nk, d) == plan


# (measured, us: 128-row kernels, key groups / one launch, 32-row kernels)
@pytest.mark.parametrize("backward,d,heads,tokens,ndocs,plan", [
    (False, 64, 12, 4096, 64, 0),   # 13.5, 30.7, 35.6
    (False, 64, 8, 1811, 31, 0),    # 10.5, 11.2, 20.2
    (False, 64, 12, 2048, 4, 1),    # 16.6, 15.6, 26.4
    (False, 128, 4, 6968, 20, 0),   # 24.3, 30.0
    (False, 64, 2, 4096, 7, 2),     # (four heads: 37.1, 31.2, 27.9)
    (False, 128, 4, 8192, 128, 0),  # 16.6, 27.7, 53.8
    (True, 64, 4, 16384, 256, 0),   # 79, 102, 122
    (True, 64, 4, 16384, 32, 0),    # 63, 74, 144
    (True, 64, 12, 4096, 64, 0),    # 49, 68, 83
    (True, 64, 4, 4096, 16, 1),     # 30.8, 17.9, 31.5
    (True, 128, 4, 8192, 64, 0),    # 42, 47, 127
    (True, 128, 1, 5115, 16, 2),    # 63, 43, 33
    (True, 64, 2, 8192, 8, 1),      # 58, 35, 44
    (True, 128, 2, 16384, 4, 1),    # 239, 184, 359
    (True, 128, 2, 4096, 2, 2),     # 129, 96, 69
    # empty documents: launches of 2^32 threads or more along one axis are refused, which 128-row kernels reach last
    (False, 64, 512, 16, 33000, 0), (True, 64, 512, 16, 33000, 0), (True, 64, 128, 129, 70000, 0)])
def test_attention_of_packed_rows_goes_by_the_length_of_the_documents(backward, d, heads, tokens, ndocs, plan):
    assert _lib.attn_plan(backward, ndocs, tokens, tokens, heads, heads, d) == plan


# (measured, us: 128 rows in two launches, in one, 32 rows)
@pytest.mark.parametrize("d,heads,b,s,plan", [
    (64, 1, 1, 16384, 2),   # 570, 353, 257
    (64, 1, 4, 8192, 1),    # 294, 181, 237
    (64, 4, 1, 16384, 0),   # 621, 609, 868
    (128, 1, 1, 16384, 2),  # 856, 705, 540
    (128, 1, 4, 8192, 1),   # 435, 368, 529
    (128, 3, 1, 12000, 1),  # 646, 546, 881
    (128, 4, 1, 16384, 0)])  # 1007, 1118, 1987
def test_attention_backward_of_long_rows(d, heads, b, s, plan):
    assert _lib.attn_plan(True, None, b * s, s, heads, heads, d) == plan


# (measured, us: 128-row kernel, 32-row kernel)
@pytest.mark.parametrize("d,heads,b,s,plan", [
    (64, 4, 1, 64, 0),    # 4.9, 5.3
    (64, 41, 3, 33, 0),   # 5.0, 5.6
    (64, 16, 4, 65, 2),   # 6.2, 5.5
    (64, 24, 4, 65, 0),   # 6.3, 6.8
    (64, 24, 4, 128, 2),  # 7.1, 7.0
    (128, 64, 2, 64, 0),  # 6.5, 7.2
    (128, 16, 1, 65, 2)])  # 7.7, 6.8
def test_attention_forward_of_short_rows(d, heads, b, s, plan):
    assert _lib.attn_plan(False, None, b * s, s, heads, heads, d) == plan


@pytest.mark.parametrize("T,h,f", [(512, 3072, 8192), (512, 4096, 11008)])
def test_a_decision_about_products_in_one_launch_is_remembered(T, h, f):
    """A layer asks several times per pass.  Where lists on 256 x 256 tiles come into question the forward form is looked up twice, with and without
    them; neither may push the other out (a repeated query then took twice as long as the weight gradients' one lookup)."""
    lib, two = _lib.load(), ctypes.c_int64 * 2
    queries = [(1, 2, two(T, T), two(f, f), h), (0, 2, two(f, f), two(h, h), T)]
    best = [float("inf")] * 2
    for _ in range(30):
        for i, q in enumerate(queries):
            start = time.perf_counter()
            for _ in range(300):
                lib.ezl_gemm_group_form_workspace_bytes(*q)
            best[i] = min(best[i], time.perf_counter() - start)
    assert best[0] <= 1.4 * best[1]


# ---- the GPU tests of single kernels reach the kernels they are about -----------------------------------------------------
FORMS = ("forward", "input gradient", "weight gradient", "weight gradient")


def listed(table):
    return [(want, case) for want, cases in table.items() for case in cases]


@pytest.mark.parametrize("want,case", listed(edges.SMALLER_TILES) + listed(edges.WIDE_TILES) + listed(edges.LARGEST_TILES))
def test_products_at_tile_edges_take_the_tiles_they_are_listed_under(want, case):
    form, M, N, K = case
    _, rows, cols, _, waves = _lib.gemm_plan(FORMS[form], [M], [N], K)
    assert (rows, cols, waves) == want


@pytest.mark.parametrize("want,case", listed(edges.PAIRS) + listed(edges.PAIRS_WIDE))
def test_products_over_pairs_take_the_tiles_they_are_listed_under(want, case):
    T, h, widths = case
    _, rows, cols, _, waves = _lib.gemm_plan("input gradient over pairs", [T], [h], sum(widths))
    assert (rows, cols, waves) == want


@pytest.mark.parametrize("T,h,widths", edges.FORWARD_LISTS)
def test_forward_products_on_the_largest_tiles_are_one_launch(T, h, widths):
    assert _lib.gemm_plan("forward", [T] * len(widths), widths, h)[:3] == (True, 256, 256)


@pytest.mark.parametrize("want,case", listed(edges.LAYER_LISTS))
def test_weight_gradients_of_a_layer_go_out_as_they_are_listed(want, case):
    h, nq, nk, f, b, s, fp32 = case
    layer = _lib.Layer(s=s, b=b, h=h, nq=nq, nk=nk, d=h // nq, f=f, ndocs=b, npos=s)
    assert _lib.layer_plan(layer, fp32) == (want is not None)
    if want:
        kv = h // nq * nk
        _, rows, cols, _, waves = _lib.gemm_plan("weight gradient", [h, kv, kv, h, f, f, h], [h] * 6 + [f], b * s)
        assert (rows, cols, waves) == want


@pytest.mark.parametrize("want,case", listed(edges.ATTENTION))
def test_attention_takes_the_kernels_it_is_listed_under(want, case):
    d, nq, nk, b, s, cu = case
    ndocs = None if cu is None else len(cu) - 1
    assert tuple(_lib.attn_plan(backward, ndocs, b * s, s, nq, nk, d) for backward in (False, True)) == want


# (measured, us, 256 x 256 against the smaller tiles whose estimate is lower)
@pytest.mark.parametrize("M,N,T,tile", [
    (50304, 1024, 1167, 256),  # 147, 175
    (70528, 2176, 477, 256),   # (bf16) 198, 221
    (151808, 1024, 711, 256),  # (bf16) 299, 319
    (11008, 4096, 1531, 256), (32000, 768, 1024, 128)])
def test_weight_gradients_of_a_vocabulary_take_smaller_tiles_only_by_a_margin(M, N, T, tile):
    assert _lib.gemm_plan("weight gradient", [M], [N], T)[1] == tile


# (form, M, N, K, shares): us in these and in the shares that the rates of operands on whole lines ask for
SHARES_OF_64 = [(0, 605, 384, 2560, 4),   # 11.2, 8 shares 12.9
                (0, 376, 576, 3328, 4),   # 11.8, 9 shares 14.0
                (1, 1551, 128, 3072, 5),  # 11.4, 10 shares 13.8
                (1, 768, 256, 4480, 5),   # 12.7, 10 shares 14.8
                (2, 576, 512, 2989, 3),   # 12.8, 7 shares 14.6
                (2, 1728, 192, 3250, 3),  # 13.3, 6 shares 15.0
                (0, 191, 320, 1728, 6),   # 9.0, whole (8 waves) 11.4
                (1, 386, 256, 1920, 6)]   # 9.6, whole 11.9


@pytest.mark.parametrize("form,M,N,K,shares", SHARES_OF_64)
def test_short_products_are_split_as_finely_as_pays(form, M, N, K, shares):
    assert _lib.gemm_plan(FORMS[form], [M], [N], K) == (True, 64, 64, shares, 4)
