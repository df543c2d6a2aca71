"""The product of a prompt's rows (``_mix.prompt_linear``) against float64, and where it is used."""

import pytest
import torch
import torch.nn.functional as F

from test_gpu_few_rows_linear import DEV, _check, _mk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 255, 256, 257, 700])
@pytest.mark.parametrize("n,k", [(8, 64), (8, 128), (248, 192), (256, 384), (264, 2048), (2064, 512)])
def test_against_float64(m, n, k):
    from astrai_amd.extension import _mix
    x, w, b = _mk(m, m, k), _mk(n, n, k, std=k ** -0.5), _mk(n + 1, n)
    exact, weight = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    _check(_mix.prompt_linear(x, w), exact, weight, 1)
    _check(_mix.prompt_linear(x, w, b), exact + b.double(), weight + b.double().abs(), 1)
    wide = _mk(5, m, k + 24)
    wide[:, 8:8 + k] = x
    assert torch.equal(_mix.prompt_linear(wide[:, 8:8 + k], w), _mix.prompt_linear(x, w))


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("m,ff,k", [(1, 8, 128), (256, 128, 256), (300, 136, 320), (257, 248, 2048), (513, 1000, 64)])
def test_activation_epilogue(act, m, ff, k):
    """The activation form is the two launches it replaces: the sums of a product run in one order."""
    from astrai_amd.extension import _mix
    x, w = _mk(m, m, k), _mk(ff, 2 * ff, k, std=k ** -0.5)
    got = _mix.prompt_linear(x, w, act=act)
    assert torch.equal(got, _mix.act_mul(_mix.prompt_linear(x, w), act))


def test_more_tiles_than_compute_units():
    """Tile counts of every remainder by eight: each tile is somebody's, and the neighbours of none."""
    from astrai_amd.extension import _mix
    w = _mk(2, 2064, 128)
    for m in (7400, 7700, 7900, 8200):
        x = _mk(m, m, 128)
        weight = x.double().abs() @ w.double().abs().t()
        _check(_mix.prompt_linear(x, w), x.double() @ w.double().t(), weight, 1)


def test_calls_that_are_left_to_the_library():
    from astrai_amd.extension import _mix, w8a8
    from astrai_amd.model import mixers
    x, w = _mk(1, 4096, 256), _mk(2, 4080, 256)
    with torch.no_grad():
        assert mixers.prompt_rows(x, w) and mixers.prompt_rows(x, w, act="silu")
        for bad in (x.float(), x.cpu(), _mk(1, 4096, 512)[:, ::2], _mk(1, 256, 4096).t()):
            assert not mixers.prompt_rows(bad, w)
        assert not mixers.prompt_rows(_mk(1, 4096, 160), _mk(2, 4080, 160)) and not mixers.prompt_rows(x, _mk(2, 4084, 256))
        assert not mixers.prompt_rows(x, _mk(2, 4096, 256)) and not mixers.prompt_rows(_mk(1, 0, 256), w)
        with w8a8.int8_autocast(True):
            assert not mixers.prompt_rows(x, w)
        with torch.autocast("cuda", dtype=torch.float16):
            assert not mixers.prompt_rows(x, w)
        assert torch.equal(mixers.linear(x, w), _mix.prompt_linear(x, w))
        mlp = mixers.GatedMLP(256, 2048).to(device=DEV, dtype=torch.bfloat16)
        mlp.gate_up.reset_parameters()
        mlp.down.reset_parameters()
        h = _mk(3, 4096, 256)
        assert torch.equal(mlp(h), F.linear(_mix.prompt_linear(h, mlp.gate_up.weight, act="silu"), mlp.down.weight))
    w.requires_grad_(True)
    assert not mixers.prompt_rows(x, w)
    mixers.linear(x, w).sum().backward()
    assert w.grad is not None
    with pytest.raises(RuntimeError, match="not covered"):
        _mix.prompt_linear(x, _mk(2, 4084, 256))
