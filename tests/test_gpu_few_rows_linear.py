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


def test_a_bias_of_another_size_is_left_to_the_library():
    """The kernels would read as many values as there are outputs."""
    from astrai_amd.extension import _mix
    from astrai_amd.model import mixers
    w = _mk(2, 264, 256)
    for x in (_mk(1, 8, 256), _mk(3, 4096, 256)):
        for bias in (_mk(4, 1), _mk(5, 263), _mk(6, 1, 264)):
            takes = bias.numel() == 264
            assert _mix.few_rows_linear_supported(x[:8], w, bias) == takes and _mix.prompt_linear_supported(x, w, bias) == takes
            if not takes:
                with pytest.raises(RuntimeError, match="not covered"):
                    _mix.few_rows_linear(x[:8], w, bias)
        with torch.no_grad():
            assert torch.equal(mixers.linear(x, w, _mk(4, 1)), F.linear(x, w, _mk(4, 1)))
            with pytest.raises(RuntimeError):
                mixers.linear(x, w, _mk(5, 263))


@pytest.mark.parametrize("parts", [1, 2, 3, 4])
@pytest.mark.parametrize("m,n,k", [(1, 64, 512), (17, 200, 128), (8, 2048, 4224), (33, 3076, 1280), (64, 132, 2048)])
def test_planes_of_ranges_add_up(parts, m, n, k):
    """Ranges without items, row ranges of one to three groups, a remainder of rows."""
    from astrai_amd.extension import _mix
    x, w = _mk(1, m, k), _mk(2, n, k)
    planes = _mix.few_rows_parts(x, w, parts)
    assert planes.shape == (parts, m, n) and planes.dtype == torch.float32
    exact, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    # fp32 sums: k + parts roundings at most, far fewer in effect
    assert ((planes.double().sum(0) - exact).abs() <= 2.0 ** -24 * (k + parts) * size).all()
    assert torch.equal(planes, _mix.few_rows_parts(x, w, parts))


@pytest.mark.parametrize("parts", [1, 2, 3, 4])
@pytest.mark.parametrize("rows,width", [(1, 33), (5, 128), (3, 1000), (9, 2048), (2, 5000), (2, 8200)])
def test_row_norms_of_planes(parts, rows, width):
    """Against the norms of the planes' sum, formed in the same order."""
    from astrai_amd.extension import _mix
    g = torch.Generator(device=DEV).manual_seed(width + parts)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    planes, x, u, w, v = rand(parts, rows, width), rand(rows, width), rand(rows, width), rand(width), rand(width)
    total = planes[0].clone()
    for p in planes[1:]:
        total += p
    for more in ({}, {"u": u}, {"vec": v, "mult": 0.5}):
        got = _mix.sum_norm(planes, w, torch.bfloat16, 1e-5, x=x, **more)
        want = _mix.sum_norm(total, w, torch.bfloat16, 1e-5, x=x, **more)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    wide = rand(parts, rows, width + 8)
    got, want = _mix.sum_norm(wide[:, :, :width], w, torch.bfloat16, 1e-5), _mix.sum_norm(wide[:, :, :width].contiguous(), w, torch.bfloat16, 1e-5)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    xs = [x.clone(), x.clone()]
    got, want = _mix.residual_norm(planes, xs[0], w, v, 0.5, 1e-5), _mix.residual_norm(total, xs[1], w, v, 0.5, 1e-5)
    assert torch.equal(xs[0], xs[1]) and torch.equal(got, want.bfloat16()) and got.dtype == torch.bfloat16
    for bad in (planes.bfloat16(), planes[:, :, :-1]):
        with pytest.raises(RuntimeError):
            _mix.sum_norm(bad, w, torch.bfloat16, 1e-5)


def test_planes_stay_between_a_layer_and_its_norm():
    """Hooks, wrappers and subclasses see the products; the model's results are those of either way."""
    from astrai_amd.model import mixers
    for n, k in ((2048, 5632), (2048, 2048)):
        assert mixers.parts_of(16, n, k) == 4
    assert mixers.parts_of(16, 4096, 4096) == mixers.parts_of(16, 2048, 1024) == 1
    mlp = mixers.GatedMLP(512, 2176)
    for product in (mlp.gate_up, mlp.down):
        product.reset_parameters()
    mlp = mlp.to(DEV).to(torch.bfloat16)
    h, seen = _mk(3, 16, 512), []
    with torch.no_grad():
        assert mixers.fed(mlp, h).shape == (4, 16, 512)
        want = mlp(h)
        assert want.shape == (16, 512)
        assert ((mixers.fed(mlp, h).sum(0) - want.float()).norm() / want.float().norm()) < 2.0 ** -8
        for module in (mlp, mlp.down):
            hook = module.register_forward_hook(lambda mod, args, out: seen.append(out.shape))
            assert mixers.fed(mlp, h).shape == (16, 512) and seen.pop() == (16, 512)
            hook.remove()

        class Other(mixers.GatedMLP):
            pass

        other = Other(512, 2176).to(DEV).to(torch.bfloat16)
        assert mixers.fed(other, h).shape == (16, 512)
