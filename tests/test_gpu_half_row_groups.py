"""8-bit products of few tokens: groups of sixteen weight rows or tokens of which 8 or fewer are there, waves with one item
of K, several or none."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
SIZES = [(1024, 256), (2048, 512), (2056, 2304), (2048, 4352), (4096, 2048), (4104, 768), (8200, 256)]


@pytest.mark.parametrize("m", [1, 2, 8, 9, 16, 17, 64, 65, 128])
@pytest.mark.parametrize("n,k", SIZES)
def test_int8_bits(m, n, k):
    from astrai_amd.extension import _cabi
    g = torch.Generator(device=DEV).manual_seed(n + m)
    a, b = (torch.randint(-15, 16, (r, k), generator=g, device=DEV, dtype=torch.int8) for r in (m, n))
    sa, sb = (torch.rand(r, generator=g, device=DEV) * 0.01 + 0.001 for r in (m, n))
    acc = a.float() @ b.float().t()   # (sums under 2^24: exact)
    assert torch.equal(_cabi.mm_int8(a, b, sa, sb), (acc * sa[:, None] * sb).bfloat16())


@pytest.mark.parametrize("m", [1, 8, 16, 33, 64, 128])
@pytest.mark.parametrize("n,k", SIZES)
def test_fp8_against_float64(m, n, k):
    """One rounding to bf16 (2^-8 of |y|, twice with the block steps' products), fp32 sums."""
    from astrai_amd.extension import _cabi
    from astrai_amd.extension.ops import fp8_block
    g = torch.Generator(device=DEV).manual_seed(n + m)
    a, b = (torch.randn(r, k, generator=g, device=DEV).to(torch.float8_e4m3fn) for r in (m, n))
    one = torch.ones(1, device=DEV)
    y, weight = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    bound = 2.0 ** -8 * y.abs() + k * 2.0 ** -23 * weight
    assert ((_cabi.mm_fp8(a, b, one, one).double() - y).abs() <= bound).all()
    if m <= 64:
        sx = torch.rand(m, k // 128, generator=g, device=DEV) + 0.5
        sw = torch.rand(-(-n // 128), k // 128, generator=g, device=DEV) + 0.5
        xd = (a.double().reshape(m, -1, 128) * sx.double()[:, :, None]).reshape(m, k)
        wd = (b.double().reshape(n, -1, 128) * sw.double()[torch.arange(n, device=DEV) // 128][:, :, None]).reshape(n, k)
        y, weight = xd @ wd.t(), xd.abs() @ wd.abs().t()
        got = fp8_block.mm_fp8_blockscaled(a, b, sx, sw).double()
        assert ((got - y).abs() <= 2.0 ** -8 * y.abs() + k * 2.0 ** -22 * weight).all()
