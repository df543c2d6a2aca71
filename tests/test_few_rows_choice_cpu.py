"""When a mixer model's product of a few rows leaves ``F.linear`` for its own kernel: not where anything besides the plain
product is asked for. The shapes and devices the kernel takes count as given here."""
import pytest
import torch

from astrai_amd.extension import _mix
from astrai_amd.model import mixers


@pytest.fixture(autouse=True)
def any_shape(monkeypatch):
    # (it looks at addresses, which wrapped and fake tensors do not have)
    monkeypatch.setattr(_mix, "few_rows_linear_supported", lambda x, w, *a, **k: bool(x.data_ptr() and w.data_ptr()))


def _operands():
    return torch.randn(4, 16), torch.randn(8, 16), torch.randn(8)


@pytest.mark.parametrize("which", range(3))
def test_gradients_of_every_operand(which):
    ops = _operands()
    assert mixers.few_rows(*ops)
    ops[which].requires_grad_(True)
    assert not mixers.few_rows(*ops)
    with torch.no_grad():
        assert mixers.few_rows(*ops)
    out = mixers.linear(*ops)
    out.sum().backward()
    assert ops[which].grad is not None


def _ways(mlp):
    """Which way ``mlp`` goes: the kernel with the activation in its epilogue, or the two modules."""
    x = torch.randn(4, 16)
    calls = []
    with pytest.MonkeyPatch.context() as m, torch.no_grad():
        m.setattr(_mix, "few_rows_linear", lambda h, w, b=None, act=None: (calls.append(act), torch.zeros(4, w.size(0) // (1 if act is None else 2)))[1])
        m.setattr(_mix, "act_mul", lambda gu, act: (calls.append("act_mul"), gu[:, :gu.size(1) // 2])[1])
        mlp(x)
    return calls


def test_the_gate_product_is_a_module_call_where_something_watches():
    mlp = mixers.GatedMLP(16, 24)
    assert _ways(mlp) == ["silu", None]
    seen = []
    for register in ("register_forward_hook", "register_forward_pre_hook"):
        hook = getattr(mlp.gate_up, register)(lambda *a: seen.append(1))
        assert _ways(mlp) == [None, "act_mul", None] and seen.pop()
        hook.remove()
    hook = torch.nn.modules.module.register_module_forward_hook(lambda *a: seen.append(1))
    try:
        assert "act_mul" in _ways(mlp) and len(seen) >= 2
    finally:
        hook.remove()
    forward, mlp.gate_up.forward = mlp.gate_up.forward, lambda x: torch.ones(4, 48)
    assert _ways(mlp) == ["act_mul", None]
    del mlp.gate_up.forward
    assert _ways(mlp) == ["silu", None]
    torch.nn.utils.parametrize.register_parametrization(mlp.gate_up, "weight", torch.nn.Identity())
    assert _ways(mlp) == [None, "act_mul", None]

    class Wrapped(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner, self.weight = inner, inner.weight

        def forward(self, x):
            return self.inner(x) + 1

    mlp = mixers.GatedMLP(16, 24)
    mlp.gate_up = Wrapped(mlp.gate_up)
    assert _ways(mlp) == [None, "act_mul", None]


def _plane_calls():
    """(what of a layer is called by the layer's forward, the call, the name under which a compiled call would run)."""
    from types import SimpleNamespace
    mlp, x = mixers.GatedMLP(16, 24), torch.randn(4, 16)
    mix = mixers.LightningAttention(16, 1, 8, 8, [0.5], 1e-5, 0)
    ctx = SimpleNamespace(parts=False)
    yield mlp, lambda: mixers.fed(mlp, x)
    yield mlp.down, lambda: mixers.rows_out(mlp.down, torch.randn(4, 24), True)
    yield mix, lambda: mixers.mixed(mix, x, ctx)
    yield mix.o, lambda: mixers.rows_out(mix.o, torch.randn(4, mix.o.weight.size(1)), True)
    yield mlp.gate_up, lambda: mlp(x)


def test_a_call_that_is_not_the_class_s_own_forward_is_made(monkeypatch):
    """Compiled modules, other forwards and other calls: none is gone around for planes or a fused product."""
    monkeypatch.setattr(mixers, "parts_of", lambda *a: 4)
    monkeypatch.setattr(_mix, "act_mul", lambda gu, act: gu[:, :gu.size(1) // 2])
    for name in ("few_rows_parts", "few_rows_linear"):
        monkeypatch.setattr(_mix, name, lambda *a, **k: pytest.fail("gone around"))
    monkeypatch.setattr(mixers, "linear", torch.nn.functional.linear)
    with torch.no_grad():
        for module, call in _plane_calls():
            seen = []

            def instead(*args):
                """``args``: of the call, or the module in front of them."""
                args = args[1:] if args[0] is module else args
                seen.append(len(args) == 1 or not args[1].parts)
                return torch.ones(4, 48)

            module.compile(backend="eager")
            module._compiled_call_impl = instead
            call()
            module._compiled_call_impl = None
            for cls, name in ((type(module), "forward"), (torch.nn.Module, "__call__")):
                with pytest.MonkeyPatch.context() as m:
                    stock = getattr(cls, name)
                    m.setattr(cls, name, lambda self, *args: (instead if self is module else stock)(self, *args))
                    call()
            assert seen == [True] * 3


def test_the_head_is_a_module_call():
    from types import SimpleNamespace
    model = mixers.MixerLM(SimpleNamespace(vocab=8, width=16), [])
    ctx, h, seen = SimpleNamespace(batch=2, seq=3), torch.randn(6, 16), []
    hook = model.head.register_forward_hook(lambda module, args, out: seen.append(args[0].shape))
    with pytest.MonkeyPatch.context() as m, torch.no_grad():
        m.setattr(_mix, "few_rows_linear", lambda x, w, b=None, act=None: x @ w.t())
        out = model.finish(h, h, ctx, torch.tensor([2]))
        assert out["logits"].shape == (2, 1, 8) and seen == [(2, 1, 16)]
        hook.remove()
        model.head = torch.nn.Sequential(torch.nn.Linear(16, 4), torch.nn.Linear(4, 5))
        assert model.finish(h, h, ctx, None)["logits"].shape == (2, 3, 5)


def test_other_handlers_of_linear_get_the_call(monkeypatch):
    from astrai_amd.extension import dispatch, fp8, w8a8
    x, w, b = _operands()
    with torch.no_grad():
        assert mixers.few_rows(x, w, b)
        with w8a8.int8_autocast(True):
            assert not mixers.few_rows(x, w, b)
        with fp8.fp8_autocast(True):
            assert not mixers.few_rows(x, w, b)
        assert mixers.few_rows(x, w, b)
        monkeypatch.setattr(dispatch, "_handlers", [*dispatch._handlers, lambda x, w, b: None])
        assert not mixers.few_rows(x, w, b)


def test_transforms_tangents_modes_and_traces():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    x, w, b = _operands()
    want = torch.nn.functional.linear(x, w, b)

    def taken(*a, **k):
        raise AssertionError("the kernel was called")

    with pytest.MonkeyPatch.context() as m, torch.no_grad():
        m.setattr(_mix, "few_rows_linear", taken)
        with pytest.raises(AssertionError):
            mixers.linear(x, w, b)
        assert torch.allclose(torch.func.vmap(lambda r: mixers.linear(r[None], w, b)[0])(x), want, atol=1e-5)
        assert torch.allclose(torch.func.vmap(lambda r: mixers.linear(x, r[None])[:, 0])(w).t(), want - b, atol=1e-5)
        assert torch.func.jvp(lambda t: mixers.linear(t, w, b), (x,), (x,))[1].shape == want.shape
        assert torch.func.grad(lambda t: mixers.linear(t, w, b).sum())(x).shape == x.shape
        with forward_ad.dual_level():
            assert forward_ad.unpack_dual(mixers.linear(forward_ad.make_dual(x, x), w, b)).tangent is not None
        with FlopCounterMode(display=False) as flops:
            mixers.linear(x, w, b)
        assert flops.get_total_flops() == 2 * 4 * 16 * 8
        with FakeTensorMode() as fake:
            mixers.linear(*(fake.from_tensor(t) for t in (x, w, b)))

        class Counting(TorchFunctionMode):
            calls = 0

            def __torch_function__(self, func, types, args=(), kwargs=None):
                self.calls += func is torch.nn.functional.linear
                return func(*args, **(kwargs or {}))

        with Counting() as mode:
            mixers.linear(x, w, b)
        assert mode.calls == 1

        class Sub(torch.Tensor):
            pass

        assert type(mixers.linear(x.as_subclass(Sub), w, b)) is Sub
        assert torch.allclose(torch.jit.trace(lambda t: mixers.linear(t, w, b), (x,), check_trace=False)(2 * x), 2 * want - b, atol=1e-5)
        assert torch.allclose(torch.compile(lambda t: mixers.linear(t, w, b), backend="eager")(x), want)


@pytest.mark.parametrize("n,k,act,most", [
    (2048, 2048, None, 64), (16384, 2048, None, 64), (16388, 2048, None, 32), (12288, 4096, None, 64), (13312, 4096, None, 32),
    (1024, 4096, None, 64), (1024, 5632, None, 32), (2048, 5632, None, 64), (32000, 2048, None, 32), (4096, 8192, None, 64),
    (8192, 8192, None, 0), (16384, 4096, "silu", 64), (16392, 4096, "silu", 32), (12288, 8192, "silu", 64), (16384, 8192, "silu", 0)])
def test_sizes_at_which_the_kernel_is_the_faster_one(n, k, act, most):
    w = torch.zeros(1).expand(n, k)
    with torch.no_grad():
        for rows in (1, 32, 33, 64, 65):
            assert mixers.few_rows(torch.zeros(1).expand(rows, k), w, act=act) == (rows <= most)


@pytest.mark.parametrize("m,n,act,taken", [
    (1024, 2 * 5632, "silu", True), (16384, 2 * 5632, "gelu_tanh", True), (1500, 2 * 5632, "silu", False),
    (4096, 3664, None, True), (5000, 3664, None, False), (4096, 4096, None, False), (2048, 6416, None, True)])
def test_prompt_sizes_at_which_the_tiles_are_the_faster_ones(monkeypatch, m, n, act, taken):
    monkeypatch.setattr(_mix, "prompt_linear_supported", lambda *a: True)
    x, w = torch.zeros(1).expand(m, 2048), torch.zeros(1).expand(n, 2048)
    with torch.no_grad():
        assert mixers.prompt_rows(x, w, act=act) == taken
    w = torch.zeros(1).expand(n, 2048).requires_grad_(True)
    assert not mixers.prompt_rows(x, w, act=act)


def test_a_prompts_products_are_taken_up_to_the_descriptors_reach():
    """Weights whose offsets stay below 2 GiB: gate and up of 32512 from 16384 values do, with 256 rows to spare."""
    lib = _mix.load()
    assert lib is not None, _mix.load_error()
    takes = lambda n, k, act, m=4096, ldx=None: bool(lib.astrai_mix_prompt_linear_takes(m, n, k, ldx or k, act))
    for n, k in ((32512, 16384), (65280, 8192), (32632, 16384)):
        assert takes(n, k, 0) and takes(n, k, 1) and takes(2 * n, k, -1), (n, k)
        assert (2 * n + 256) * k * 2 < 2 ** 31
    assert not takes(32640, 16384, 0) and not takes(65280, 16384, -1)
    assert not takes(2 ** 22, 64, -1) and takes(2 ** 22 - 8, 64, -1)
    assert takes(64, 16384, -1, 2 ** 16 - 257) and not takes(64, 16384, -1, 2 ** 16 - 256)
    assert not takes(64, 64, -1, 2 ** 40) and not takes(64, 2 ** 40, -1) and not takes(2 ** 40, 64, -1)
    assert not takes(60, 64, -1) and not takes(64, 96, -1) and not takes(64, 128, -1, ldx=120) and not takes(64, 128, -1, ldx=132)
    assert not takes(64, 64, -1, 0)
