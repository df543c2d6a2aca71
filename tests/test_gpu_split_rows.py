"""Products whose rows are split over two tile sizes, against the accumulators of the unsplit kernels."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _fp8(seed, r, c, dtype=torch.float8_e4m3fn):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(r, c, generator=g, device=DEV).to(dtype)


@pytest.mark.parametrize("m,n,k", [(2816, 4096, 256), (4300, 4096, 256), (4300, 4096, 384), (4601, 4096, 128 * 3),
                                   (3001, 11264, 256), (5500, 3080, 256), (520, 65544, 256)])
def test_split_rows_give_the_unsplit_bits(m, n, k):
    """int8: the same integers whatever tile a row falls on. fp8: a row's sum in the same order of K in every
    tile kernel up to fp32 rounding: both round to bf16 once (2^-8 of |y| for one ulp, sums good to 6e-5 of their rms)."""
    from astrai_amd.extension import _cabi
    g = torch.Generator(device=DEV).manual_seed(m)
    a = torch.randint(-127, 128, (m, k), generator=g, device=DEV, dtype=torch.int8)
    b = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
    sa, sb = torch.rand(m, generator=g, device=DEV) + 0.5, torch.rand(n, generator=g, device=DEV) + 0.5
    got = _cabi.mm_int8(a, b, sa, sb)
    acc = _cabi.mm_int8(a, b, None, None, None, 2)
    assert torch.equal(got, (acc.float() * sa[:, None] * sb[None, :]).to(torch.bfloat16)), _cabi.last_kernel()
    rows = torch.tensor([0, m // 2, m - 1], device=DEV)
    assert torch.equal(acc[rows].double(), a[rows].double() @ b.double().t())
    fa, fb = _fp8(m, m, k), _fp8(n, n, k)
    s = torch.ones(1, device=DEV)
    out, want = _cabi.mm_fp8(fa, fb, s, s).float(), _cabi.mm_fp8_acc(fa, fb)
    bound = 2.0 ** -8 * want.abs() + 2 * 8e-5 * want.square().mean().sqrt()
    assert ((out - want).abs() <= bound).all(), _cabi.last_kernel()
    assert torch.equal(_cabi.mm_fp8(fa, fb, sa * 0 + 1, sb * 0 + 1).float(), out)   # one step per row and column: ones
