"""Products on 192 x 256 tiles, short reductions on the 4-wave kernel and half a chip's worth of tiles in two shares, each against fp32."""
import ctypes

import pytest
import torch

from easyllm_amd import _lib
from test_kernel_edges_gpu import K, check_gemm, gemm_bound, products, rnd  # noqa: F401

FORMS = ("forward", "input gradient", "weight gradient", "weight gradient")
# (form, M, N, K) by (tile rows, columns, waves, shares of a reduction in the last round); forms as in check_gemm
TILES = {
    # two and more K tiles, ragged rows, one round and several
    (192, 256, 4, 1): [(0, 2100, 4096, 128), (0, 6000, 3072, 128), (1, 1531, 6144, 128), (0, 3664, 2368, 2048), (0, 2303, 8192, 128), (2, 3008, 3072, 1105),
                       (2, 3008, 6144, 1169), (3, 2304, 4096, 1105)],
    # the last round's tiles in shares, with a K tail
    (192, 256, 4, 5): [(0, 700, 3072, 8192), (1, 2100, 1024, 8192), (2, 1536, 1536, 9233), (3, 768, 3072, 9233)],
    (192, 256, 4, 2): [(0, 1500, 4096, 11008), (1, 1531, 4096, 11008)],
    # half the chip in two shares; one round of a short weight gradient
    (256, 256, 4, 2): [(1, 4000, 2048, 32000), (0, 2048, 4096, 20032)],
    (256, 256, 4, 1): [(2, 4096, 4096, 1531), (3, 4096, 4096, 1100)]}


@pytest.mark.gpu
@pytest.mark.parametrize("want,case", [(w, c) for w, cs in TILES.items() for c in cs])
def test_products_on_large_tiles(K, want, case):  # noqa: F811
    print("gemm", want, case, flush=True)
    form, M, N, Kd = case
    check_gemm(K, form, M, N, Kd)
    check_gemm(K, form, M, N, Kd, accumulate=True, seed=5)
    if form == 0:  # bf16 values in fp32: the same sums, rounded the same way
        x, w = rnd(M, Kd, seed=1), rnd(N, Kd, seed=2)
        assert torch.equal(K.linear_fwd(x, w, fp32_output=True), K.linear_fwd(x, w).float())


@pytest.mark.parametrize("want,case", [(w, c) for w, cs in TILES.items() for c in cs])
def test_products_take_the_large_tiles_they_are_listed_under(want, case):
    form, M, N, Kd = case
    _, rows, cols, split, waves = _lib.gemm_plan(FORMS[form], [M], [N], Kd)
    assert (rows, cols, waves, split) == want


PAIRS = [(1531, 4096, (5504, 5504)), (2100, 4096, (72, 56)), (1531, 4096, (4096, 3464, 3448))]


@pytest.mark.gpu
@pytest.mark.parametrize("T,n_in,outs", PAIRS)
def test_input_gradient_over_pairs_on_large_tiles(K, T, n_in, outs):  # noqa: F811
    """Whole K tiles, and K tails inside the reduction."""
    print("dgrad multi", T, n_in, outs, flush=True)
    ld = max(outs)
    dys = [torch.empty(T, ld, device="cuda", dtype=torch.bfloat16)[:, :o].copy_(rnd(T, o, seed=i)) for i, o in enumerate(outs)]
    ws = [rnd(o, n_in, seed=10 + i) for i, o in enumerate(outs)]
    A, B = torch.cat([d.contiguous() for d in dys], 1), torch.cat(ws, 0)
    ref = A.float() @ B.float()
    dx = K.linear_dgrad_multi(dys, ws)
    assert ((dx.float() - ref).abs() <= gemm_bound(A, B) + ref.abs() * 2.0 ** -8 + 1e-6).all()


@pytest.mark.parametrize("T,n_in,outs", PAIRS)
def test_pairs_take_the_large_tiles(T, n_in, outs):
    assert _lib.gemm_plan("input gradient over pairs", [T], [n_in], sum(outs))[1:3] == (192, 256)


# K tails that make the pairs' K tiles, rounded up one by one, enough for one share more than the workspace is for
@pytest.mark.gpu
@pytest.mark.parametrize("T,n_in,outs", [(201, 768, (21032, 17816)), (214, 256, (19480, 10192, 20952))])
def test_pairs_with_tails_are_split_as_their_workspace_says(K, T, n_in, outs):  # noqa: F811
    """The workspace that is asked for is enough for the plan: more of it changes no bit (a reduction that is not split is another sum)."""
    print("dgrad multi, shares", T, n_in, outs, flush=True)
    rows, cols, split = _lib.gemm_plan("input gradient over pairs", [T], [n_in], sum(outs))[1:4]
    tiles = (T + rows - 1) // rows * ((n_in + cols - 1) // cols)
    need = _lib.gemm_workspace_bytes(T, n_in, sum(outs))
    assert split > 64 and need == tiles * split * rows * cols * 4 and sum((o + 63) // 64 for o in outs) // 8 == split + 1
    dys = [rnd(T, max(outs), seed=i)[:, :o] for i, o in enumerate(outs)]
    ws = [rnd(o, n_in, seed=10 + i) for i, o in enumerate(outs)]
    n = len(outs)
    ptrs, got = ctypes.c_void_p * n, []
    for size in (need, 2 * need):
        room, dx = torch.empty(size, dtype=torch.uint8, device="cuda"), torch.empty(T, n_in, dtype=torch.bfloat16, device="cuda")
        _lib.call("ezl_gemm_bf16_ksplit", n, ptrs(*[d.data_ptr() for d in dys]), ptrs(*[w.data_ptr() for w in ws]), dx.data_ptr(), T, n_in,
                  (ctypes.c_int64 * n)(*outs), max(outs), n_in, n_in, 1, 0, 0, 0, room.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
        got.append(dx)
    assert torch.equal(*got)
    A, B = torch.cat([d.contiguous() for d in dys], 1), torch.cat(ws, 0)
    ref = A.float() @ B.float()
    assert ((got[0].float() - ref).abs() <= gemm_bound(A, B) + ref.abs() * 2.0 ** -8 + 1e-6).all()


# (form, M, N, K, shares): every count of partial tiles that are added at a time (8, 4, 2, 1), edges inside the last vector
SHARES = [(0, 2048, 2304, 8192, 3), (0, 1500, 1800, 32768, 5), (0, 1500, 1536, 32768, 7), (0, 1024, 1280, 32768, 12), (1, 1167, 2048, 32768, 6),
          (2, 2048, 1800, 16445, 4), (2, 904, 1800, 32829, 8)]


@pytest.mark.gpu
@pytest.mark.parametrize("form,M,N,Kd,shares", SHARES)
def test_partial_tiles_are_added(K, form, M, N, Kd, shares):  # noqa: F811
    """Whole vectors, and results of which no row but the first starts on 16 bytes: element by element, the same bits."""
    print("gemm shares", form, M, N, Kd, flush=True)
    check_gemm(K, form, M, N, Kd)
    check_gemm(K, form, M, N, Kd, accumulate=True, seed=5)
    A, B = rnd(M, Kd) if form < 2 else rnd(Kd, M), rnd(N, Kd, seed=1) if form == 0 else rnd(Kd, N, seed=1)
    wide = torch.zeros(M, N + 1, device="cuda", dtype=torch.float32 if form == 2 else torch.bfloat16)
    args = A, B, M, N, Kd, A.stride(0), B.stride(0), form < 2, form == 0
    K.gemm(*args, out=wide[:, :N])
    assert torch.equal(wide[:, :N], K.gemm(*args, out=torch.zeros_like(wide)[:, 1:].contiguous())) and not wide[:, N].any()


@pytest.mark.parametrize("form,M,N,Kd,shares", SHARES)
def test_products_are_split_as_they_are_listed(form, M, N, Kd, shares):
    assert _lib.gemm_plan(FORMS[form], [M], [N], Kd)[1:4] == (256, 256, shares)
