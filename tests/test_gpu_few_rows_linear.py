"""The decode-step product of the mixer models (``_mix.few_rows_linear``) against float64, and where it is used."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _mk(seed, *size, std=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*size, generator=g, device=DEV) * std).to(torch.bfloat16)


def _check(got, want, weight, rounds):
    """``rounds`` roundings to bf16 (2^-8 of |y| each), fp32 sums of k products in any order
    (k 2^-24 of the sum of their magnitudes at the very most, taken at k = 5632)."""
    bound = rounds * 2.0 ** -8 * want.abs() + 5632 * 2.0 ** -24 * weight
    err = (got.double() - want).abs()
    assert torch.isfinite(got).all() and (err <= bound).all(), (err / bound.clamp_min(1e-30)).max().item()


@pytest.mark.parametrize("m", [1, 2, 15, 16, 17, 32, 33, 48, 64])
@pytest.mark.parametrize("n,k", [(4, 128), (20, 256), (2048, 128), (1028, 384), (2052, 2048), (4100, 1152), (12292, 256),
                                 (13000, 128)])
def test_against_float64(m, n, k):
    from astrai_amd.extension import _mix
    x, w, b = _mk(m, m, k), _mk(n, n, k, std=k ** -0.5), _mk(n + 1, n)
    exact, weight = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    _check(_mix.few_rows_linear(x, w), exact, weight, 1)
    _check(_mix.few_rows_linear(x, w, b), exact + b.double(), weight + b.double().abs(), 1)
    _check(_mix.few_rows_linear(x, w, out_dtype=torch.float32), exact, weight + exact.abs(), 0)
    # x as columns of a wider matrix
    wide = _mk(5, m, k + 24)
    wide[:, 8:8 + k] = x
    assert torch.equal(_mix.few_rows_linear(wide[:, 8:8 + k], w), _mix.few_rows_linear(x, w))


@pytest.mark.parametrize("m", [1, 8, 9])
@pytest.mark.parametrize("n,k", [(1024, 3968), (1024, 4096), (2048, 4224), (2044, 4736), (2052, 4096), (2048, 5632), (5636, 1024),
                                 (6148, 256)])
def test_half_groups_and_one_or_two_items_under_way(m, n, k):
    """8 rows or tokens and fewer of a group of sixteen, one more; every remainder of the walk over a wave's items."""
    from astrai_amd.extension import _mix
    x, w = _mk(m, m, k), _mk(n, n, k, std=k ** -0.5)
    _check(_mix.few_rows_linear(x, w), x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t(), 1)


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("m,ff,k", [(1, 8, 128), (3, 5632, 256), (17, 104, 384), (32, 4104, 1152), (64, 8200, 128)])
def test_activation_epilogue(act, m, ff, k):
    """The activation form is the two launches it replaces wherever both products round alike; elsewhere a bf16
    ulp of a factor apart (|d act(z)| < 1.2 |dz|)."""
    from astrai_amd.extension import _mix
    x, w = _mk(m, m, k), _mk(ff, 2 * ff, k, std=k ** -0.5)
    got = _mix.few_rows_linear(x, w, act=act)
    gu = _mix.few_rows_linear(x, w)
    assert torch.equal(got, _mix.act_mul(gu, act))   # (the same split of K at these sizes)
    g, u = (x.double() @ w.double().t()).chunk(2, -1)
    want = (F.silu(g) if act == "silu" else F.gelu(g, approximate="tanh")) * u
    bound = 2.0 ** -8 * (1.2 * g.abs() * u.abs() + 2 * want.abs()) + 1e-5 * (1 + g.abs() + u.abs())
    assert ((got.double() - want).abs() <= bound).all()


def test_calls_that_are_left_to_the_library():
    from astrai_amd.extension import _mix, w8a8
    from astrai_amd.model import mixers
    x, w = _mk(1, 8, 256), _mk(2, 64, 256)
    with torch.no_grad():
        assert mixers.few_rows(x, w)
        for bad in (_mk(1, 65, 256), _mk(1, 8, 256).float(), x.cpu(), _mk(1, 8, 512)[:, ::2], _mk(1, 9, 256)[1:, :].t()):
            assert not mixers.few_rows(bad, w)
        assert not mixers.few_rows(_mk(1, 8, 192), _mk(2, 64, 192)) and not mixers.few_rows(x, _mk(2, 66, 256))
        assert not mixers.few_rows(x, w, torch.zeros(64, device=DEV)) and not mixers.few_rows(_mk(1, 0, 256), w)
        with w8a8.int8_autocast(True):
            assert not mixers.few_rows(x, w)
        with torch.autocast("cuda", dtype=torch.float16):
            assert not mixers.few_rows(x, w)
    w.requires_grad_(True)
    assert not mixers.few_rows(x, w)
    mixers.linear(x, w).sum().backward()
    assert w.grad is not None
    with pytest.raises(RuntimeError, match="not covered"):
        _mix.few_rows_linear(_mk(1, 65, 256), w)
