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
