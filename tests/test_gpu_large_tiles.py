"""8-bit products on the 256 x 256 and 128 x 128 tiles: even and odd numbers of K slabs, ragged edges, tile counts of every kind."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _codes(seed, rows, k):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(-127, 128, (rows, k), generator=g, device=DEV, dtype=torch.int8)


@pytest.mark.parametrize("m,n,k", [(3585, 3720, 256), (3500, 3592, 384), (4096, 4096, 640), (8200, 1800, 896)])
def test_int8_bits(m, n, k):
    """bf16 of the exact sum times both steps, rounded product by product (and once more for bias and residual)."""
    from astrai_amd.extension import _cabi
    a, b = _codes(m, m, k), _codes(n, n, k)
    g = torch.Generator(device=DEV).manual_seed(1)
    sa, sb = (torch.rand(r, generator=g, device=DEV) * 0.01 + 0.001 for r in (m, n))
    bias, resid = (torch.randn(*s, generator=g, device=DEV).bfloat16() for s in ((n,), (m, n)))
    acc = (a.float() @ b.float().t())   # (sums under 2^24: exact)
    y = acc * sa[:, None] * sb
    assert torch.equal(_cabi.mm_int8(a, b, sa, sb), y.bfloat16())
    assert "wave128" in _cabi.last_kernel()
    assert torch.equal(_cabi.mm_int8(a, b, sa, sb, bias), (y + bias.float()).bfloat16())
    assert torch.equal(_cabi.mm_int8_resid(a, b, sa, sb, resid), (y.bfloat16().float() + resid.float()).bfloat16())


@pytest.mark.parametrize("fmt", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("m,n,k", [(3585, 3720, 256), (3500, 3592, 384), (4096, 4096, 640)])
def test_fp8_against_float64(fmt, m, n, k):
    """One rounding to bf16 (2^-8 of |y|), fp32 sums; bias before or behind a rounding."""
    from astrai_amd.extension import _cabi
    g = torch.Generator(device=DEV).manual_seed(k)
    a, b = (torch.randn(r, k, generator=g, device=DEV).to(fmt) for r in (m, n))
    sa, sb = (torch.rand(1, generator=g, device=DEV) + 0.5 for _ in range(2))
    bias = torch.randn(n, generator=g, device=DEV).bfloat16()
    step = (sa.double() * sb.double()).item()
    y, weight = a.double() @ b.double().t() * step, a.double().abs() @ b.double().abs().t() * step
    slack = 2.0 ** -8 * y.abs() + k * 2.0 ** -23 * weight
    for extra, kw in ((0.0, {}), (bias.double(), dict(bias=bias)), (bias.double(), dict(bias=bias, round_first=True))):
        got = _cabi.mm_fp8(a, b, sa, sb, **kw).double()
        want = y + extra
        assert ((got - want).abs() <= slack + 2.0 ** -8 * want.abs()).all(), kw


@pytest.mark.parametrize("m,n,k", [(1100, 4096, 512), (4300, 4096, 256), (2570, 2056, 384), (6000, 1536, 256), (1500, 7168, 256)])
def test_block_scales_against_float64(m, n, k):
    """The 128-block product where it moves to large tiles, and where its last rows go out on smaller ones."""
    from astrai_amd.extension.ops import fp8_block
    g = torch.Generator(device=DEV).manual_seed(m)
    x = (torch.randn(m, k, generator=g, device=DEV) * torch.rand(m, 1, generator=g, device=DEV)).bfloat16()
    w = (torch.randn(n, k, generator=g, device=DEV) * 0.1).bfloat16()
    (x8, sx), (w8, sw) = fp8_block.quantize_act_block128(x), fp8_block.quantize_weight_block128(w)
    xd = x8.double().reshape(m, k // 128, 128) * sx.double().reshape(m, k // 128, 1)
    rows = torch.arange(n, device=DEV) // 128
    wd = w8.double().reshape(n, k // 128, 128) * sw.double().reshape(-1, k // 128)[rows][:, :, None]
    want = xd.reshape(m, k) @ wd.reshape(n, k).t()
    weight = xd.abs().reshape(m, k) @ wd.abs().reshape(n, k).t()
    got = fp8_block.mm_fp8_blockscaled(x8, w8, sx, sw).double()
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + k * 2.0 ** -23 * weight).all()


@pytest.mark.parametrize("m,n,k", [(1100, 4096, 512), (2570, 2056, 384), (4300, 4096, 256), (4096, 4096, 640)])
def test_block_steps_of_any_sign_and_size(m, n, k):
    """Negative, zero and NaN steps, steps as small as the quantizers give, and all of them beside ordinary ones in a row."""
    from astrai_amd.extension import _cabi
    g = torch.Generator(device=DEV).manual_seed(m)
    a, b = (torch.randn(r, k, generator=g, device=DEV).to(torch.float8_e4m3fn) for r in (m, n))
    sa = (torch.rand(m, k // 128, generator=g, device=DEV) + 0.5) * 1e-2
    sb = (torch.rand(-(-n // 128), k // 128, generator=g, device=DEV) + 0.5) * 1e-2
    least = 1e-12 / 448
    sa[::3] *= -1
    sb[1] *= -1
    sa[5::7, 0] = sa[6::7, -1] = least     # in front of and behind ordinary steps,
    sa[8::16] = least                      # in whole rows,
    sb[2] = sb[-1, 0] = least              # and with the weights'
    sa[9::32, 1] = 0.0
    nan_rows, nan_block = slice(10, None, 64), 3
    sa[nan_rows, 1] = sb[nan_block, 0] = float("nan")
    cols = torch.arange(n, device=DEV) // 128
    xd = a.double().reshape(m, -1, 128) * sa.double()[:, :, None]
    wd = b.double().reshape(n, -1, 128) * sb.double()[cols][:, :, None]
    xd, wd = xd.reshape(m, k), wd.reshape(n, k)
    want, weight = xd @ wd.t(), xd.abs() @ wd.abs().t()
    got = _cabi.mm_fp8_block128(a, b, sa, sb).double()
    nan = torch.zeros(m, n, device=DEV, dtype=torch.bool)
    nan[nan_rows], nan[:, cols == nan_block] = True, True
    assert torch.equal(got.isnan(), nan)
    # (a zero step counts as 1e-15, the others are at most 0.015, codes of 448)
    slack = 2.0 ** -8 * want.abs() + k * 2.0 ** -23 * weight + (k // 128) * 1.5e-17 * 128 * 448.0 ** 2 * (sa == 0).any(1, keepdim=True)
    assert (((got - want).abs() <= slack) | nan).all()
    assert (got[8] != 0).any() and (got[8, cols == 2].abs().max() < 1e-20)


# (264 tiles: those of 128 x 256 take them; 399, which are more than a round of those too, have two workgroups to a unit)
@pytest.mark.parametrize("m,n", [(185, 9000), (1500, 1536), (2048, 2040), (1300, 3072), (17000, 384), (17000, 380)])
@pytest.mark.parametrize("k", [128, 256, 384, 512, 640, 768, 896, 1024])
def test_128_tiles_of_one_and_of_two_workgroups_a_unit(m, n, k):
    """One to eight slabs, on two LDS stages and on four; one workgroup to a compute unit and more."""
    from astrai_amd.extension import _cabi
    a, b = _codes(m, m, k), _codes(n, n, k)
    g = torch.Generator(device=DEV).manual_seed(1)
    sa, sb = (torch.rand(r, generator=g, device=DEV) * 0.01 + 0.001 for r in (m, n))
    acc = (a.float() @ b.float().t())   # (sums under 2^24: exact)
    assert torch.equal(_cabi.mm_int8(a, b, sa, sb), (acc * sa[:, None] * sb).bfloat16())
    assert _cabi.last_kernel() == ("mid128x256" if (m, n) == (1300, 3072) else "mid128")
    one, bias = torch.ones(1, device=DEV), torch.randn(n, generator=g, device=DEV).bfloat16()
    a8, b8 = ((t.float() / 16).to(torch.float8_e4m3fn) for t in (a, b))
    y, weight = a8.double() @ b8.double().t(), a8.double().abs() @ b8.double().abs().t()
    for extra, kw in ((0.0, {}), (bias.double(), dict(bias=bias, round_first=True))):
        want = y + extra
        bound = 2.0 ** -8 * (y.abs() + want.abs()) + k * 2.0 ** -23 * weight
        assert ((_cabi.mm_fp8(a8, b8, one, one, **kw).double() - want).abs() <= bound).all()
