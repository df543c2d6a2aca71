"""The fp8 product with a bias added to its rounded output, against the separate operations it replaces."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _fp8(seed, r, c, dtype=torch.float8_e4m3fn):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(r, c, generator=g, device=DEV).to(dtype)


# (m, n, k) -> the kernels: decode rows, 64 and 128 tiles, large tiles (even and odd slab counts, whole rounds, tails),
# other tile kernels (n % 8, k % 128), the any-shape kernel
SHAPES = [(1, 260, 256), (100, 516, 512), (300, 1000, 384), (1100, 2056, 256), (3001, 4104, 256), (3000, 4096, 384),
          (2900, 6000, 128), (3000, 4100, 256), (200, 300, 144), (37, 50, 40)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("fmt", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_bias_after_the_rounding_is_the_separate_addition(m, n, k, fmt):
    from astrai_amd.extension import _cabi
    a, b = _fp8(m, m, k, fmt), _fp8(n, n, k, fmt)
    s = torch.tensor([0.037], device=DEV)
    bias = torch.randn(n + 1, generator=torch.Generator(device=DEV).manual_seed(k), device=DEV).to(torch.bfloat16)
    for bb in (bias[:n], bias[1:]):   # (the second starts at an odd element)
        want = _cabi.mm_fp8(a, b, s, s) + bb
        got = _cabi.mm_fp8(a, b, s, s, 0, None, bb, True)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), _cabi.last_kernel()
    nan = bias[:n].clone()
    nan[0], nan[-1] = float("nan"), float("inf")
    got = _cabi.mm_fp8(a, b, s, s, 0, None, nan, True)
    assert got[:, 0].isnan().all() and got[:, -1].isinf().all() and torch.isfinite(got[:, 1:-1]).all()


def test_dynamic_forward_with_a_bias():
    import torch.nn.functional as F
    from astrai_amd.extension import fp8
    g = torch.Generator(device=DEV).manual_seed(2)
    x = torch.randn(3, 67, 512, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(264, 512, generator=g, device=DEV).to(torch.bfloat16)
    b = torch.randn(264, generator=g, device=DEV)
    with torch.no_grad(), fp8.fp8_autocast(True, recipe=fp8.DynamicScaling()):
        plain = F.linear(x, w)
        assert torch.equal(F.linear(x, w, b.to(torch.bfloat16)), plain + b.to(torch.bfloat16))
        # a bias of another type is added as before, with the type promotion that has
        wide = fp8.fp8_linear_forward(x, w, b)
        assert wide.dtype == torch.float32 and torch.equal(wide, plain + b)
    fp8.fp8_state().reset()


def test_a_direct_forward_keeps_the_bias_gradient():
    """The function itself stands above autograd: under dynamic scaling the bias is added to the finished product."""
    from astrai_amd.extension import fp8
    g = torch.Generator(device=DEV).manual_seed(3)
    x, w, b = (torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16) for s in ((33, 256), (40, 256), (40,)))
    with fp8.fp8_autocast(True, recipe=fp8.DynamicScaling()):
        out = fp8.fp8_linear_forward(x, w, b.requires_grad_(True))
        out.backward(torch.ones_like(out))
        assert torch.equal(b.grad, torch.full_like(b, 33))
        with torch.no_grad():
            assert torch.equal(torch.nn.functional.linear(x, w, b), out)
    fp8.fp8_state().reset()
