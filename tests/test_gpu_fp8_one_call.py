"""The fp8 policy's forward and backward as one library call each against its general path: the same outputs, gradients,
histories and steps, bit for bit."""

import pytest
import torch
import torch.nn.functional as F

from astrai_amd.extension import fp8

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def fresh():
    fp8.fp8_state().reset()
    yield
    fp8.fp8_state().reset()


def _mk(seed, *size, std=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*size, generator=g, device=DEV) * std).bfloat16()


def _steps(monkeypatch, general, recipe, shape, n, bias, grads, fmt, cache):
    calls = []
    take = fp8.linear_fp8_takes
    monkeypatch.setattr(fp8, "linear_fp8_takes", lambda *a: not general and (calls.append(take(*a)) or calls[-1]))
    fp8.fp8_state().reset()
    k = shape[-1]
    w, b = _mk(1, n, k, std=0.02), _mk(2, n) if bias else None
    if grads:
        w.requires_grad_(True)
    out = []
    with fp8.fp8_autocast(True, recipe=recipe(), fp8_format=fmt):
        fp8.fp8_cache_weights(cache)
        for t in range(4):
            x = _mk(10 + t, *shape, std=1.0 + t).requires_grad_(grads)
            with torch.set_grad_enabled(grads):
                y = F.linear(x, w, b)
            out.append(y.detach())
            if grads:
                out += torch.autograd.grad(y, [x, w], _mk(20 + t, *y.shape, std=0.01))
        meta = fp8.fp8_state().peek_weight_meta(w)
        out += [r for ring in (meta._x, meta._w, meta._g) for r in (ring.hist, ring.scale, torch.tensor(ring.idx))]
    monkeypatch.setattr(fp8, "linear_fp8_takes", take)
    return out, calls


@pytest.mark.parametrize("recipe", [lambda: fp8.DelayedScaling(history_len=3, margin=1), fp8.DynamicScaling])
@pytest.mark.parametrize("shape,n,bias", [((1, 256), 256, False), ((3, 5, 512), 512, True), ((100, 272), 272, True),
                                          ((1037, 1024), 1024, False), ((64, 64, 256), 264, True)])
@pytest.mark.parametrize("grads,fmt,cache", [(False, "hybrid", None), (False, "e5m2", False), (True, "hybrid", None),
                                             (True, "e4m3", True)])
def test_same_as_the_general_path(monkeypatch, recipe, shape, n, bias, grads, fmt, cache):
    got, calls = _steps(monkeypatch, False, recipe, shape, n, bias, grads, fmt, cache)
    want, none = _steps(monkeypatch, True, recipe, shape, n, bias, grads, fmt, cache)
    # four forwards, and behind each (square weights) the input and the gradient of a backward
    assert all(calls) and len(calls) == (12 if grads and n == shape[-1] else 4) and not none
    for a, b in zip(got, want, strict=True):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


# one workgroup and part of the next, the limits of the quantizers that measure or push by themselves, just past them
@pytest.mark.parametrize("recipe", [lambda: fp8.DelayedScaling(history_len=3, margin=1), fp8.DynamicScaling])
@pytest.mark.parametrize("rows", [1, 512, 513, 1025, 2048, 2049, 4097, 8192, 8193])
def test_few_values(monkeypatch, recipe, rows):
    got, calls = _steps(monkeypatch, False, recipe, (rows, 16), 64, True, False, "hybrid", True)
    want, none = _steps(monkeypatch, True, recipe, (rows, 16), 64, True, False, "hybrid", True)
    assert all(calls) and len(calls) == 4 and not none
    for a, b in zip(got, want, strict=True):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("rows", [1, 100])   # pushed in the quantizer's launch, behind the product
def test_a_step_that_two_operands_share(rows):
    """One tensor as the step of x and of the weight's codes: the product reads it before it is refreshed."""
    from astrai_amd.extension import _cabi
    x, w, got = _mk(1, rows, 512, std=3.0), _mk(2, 64, 512), []
    codes = (w.float() / 0.01).clamp(-448, 448).to(torch.float8_e4m3fn)
    for shared in (False, True):
        sx, hist = torch.full((1,), 0.01, device=DEV), torch.ones(4, device=DEV)
        out = _cabi.linear_fp8(x, w, None, codes, (sx, sx if shared else sx.clone()), ((hist, 1), None), 0, 448.0, 1.0)
        got.append((out, sx, hist))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and got[1][1] != 0.01


@pytest.mark.parametrize("recipe", [lambda: fp8.DelayedScaling(history_len=3, margin=1), fp8.DynamicScaling])
@pytest.mark.parametrize("m,n,k", [(1, 64, 512), (48, 512, 256), (100, 272, 1024), (130, 1040, 272), (1037, 256, 512)])
@pytest.mark.parametrize("bias,fmt", [(False, "hybrid"), (True, "hybrid"), (True, "e4m3")])
def test_backward_of_weights_that_are_not_square(monkeypatch, recipe, m, n, k, bias, fmt):
    """Called directly: the gradient's handler takes square weights only."""
    one = {name: getattr(fp8, name) for name in ("_forward_in_one_call", "_backward_in_one_call")}
    results = []
    for general in (False, True):
        fp8.fp8_state().reset()
        took = []
        for name, call in one.items():
            monkeypatch.setattr(fp8, name, lambda *a, call=call: (took.append(None if general else call(*a)), took[-1])[1])
        w, out = _mk(1, n, k, std=0.02), []
        with torch.no_grad(), fp8.fp8_autocast(True, recipe=recipe(), fp8_format=fmt):
            for t in range(4):
                x, g = _mk(10 + t, m, k, std=1.0 + t), _mk(20 + t, m, n, std=0.01)
                out.append(fp8.fp8_linear_forward(x, w, None, True))
                grads = fp8.fp8_linear_backward(g, x, w, [True, True, bias])
                assert [tuple(t.shape) for t in grads] == [(m, k), (n, k), (n if bias else 0,)]
                out += grads
            meta = fp8.fp8_state().peek_weight_meta(w)
        out += [r for ring in (meta._x, meta._w, meta._g) for r in (ring.hist, ring.scale, torch.tensor(ring.idx))]
        assert len(took) == 8 and all((r is None) == general for r in took)
        results.append(out)
    for a, b in zip(*results, strict=True):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


def test_operands_that_are_left_to_the_general_path():
    from astrai_amd.extension.ops.fp8 import linear_fp8_takes
    x, w = _mk(1, 8, 256), _mk(2, 64, 256)
    assert linear_fp8_takes(x, w, None) and linear_fp8_takes(x, w, _mk(3, 64))
    for bad in (_mk(1, 8, 512)[:, ::2], _mk(1, 256, 8).t(), x.float(), x.cpu(), _mk(1, 0, 256), _mk(1, 9 * 256)[1:2049].reshape(8, 256)):
        assert not linear_fp8_takes(bad, w, None)
    assert not linear_fp8_takes(_mk(1, 8, 250), _mk(2, 64, 250), None)
    for bad in (_mk(3, 64).float(), _mk(3, 1, 64), _mk(3, 128)[::2]):
        assert not linear_fp8_takes(x, w, bad)
    for recipe in (fp8.DynamicScaling(), fp8.DelayedScaling()):   # rows of another width: refused, as by the general path
        for bad in (_mk(1, 8, 512), _mk(1, 8, 128)):
            assert not linear_fp8_takes(bad, w, None)
            with torch.no_grad(), fp8.fp8_autocast(True, recipe=recipe), pytest.raises(RuntimeError):
                fp8.fp8_linear_forward(bad, w, None, True)


def test_infinities_and_nan_reach_the_step_alike(monkeypatch):
    """A maximum passes NaN by and keeps an infinity, on both paths."""
    for value in (float("inf"), float("nan")):
        outs = []
        for general in (False, True):
            fp8.fp8_state().reset()
            take = fp8.linear_fp8_takes
            monkeypatch.setattr(fp8, "linear_fp8_takes", lambda *a: not general and take(*a))
            x, w = _mk(1, 40, 256), _mk(2, 64, 256)
            x[3, 7] = value
            with torch.no_grad(), fp8.fp8_autocast(True, recipe=fp8.DynamicScaling()):
                outs.append(F.linear(x, w))
            monkeypatch.setattr(fp8, "linear_fp8_takes", take)
        assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


def test_replayed_in_a_graph():
    x, w = _mk(1, 40, 256), _mk(2, 64, 256)
    with torch.no_grad(), fp8.fp8_autocast(True, recipe=fp8.DynamicScaling()):
        F.linear(x, w)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = F.linear(x, w)
        for t in range(4):
            x.copy_(_mk(30 + t, 40, 256, std=1.0 + t))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, F.linear(x, w))
