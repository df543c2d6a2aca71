"""The native form of the adapters' everyday calls: what it does not take is left to the adapters (which say what is wrong),
and what it takes gives the bits that their own path gives."""
import os
import subprocess
import sys

import pytest
import torch

from astrai_amd.extension import _cabi, _mix

BF16 = torch.bfloat16


class Refuses:
    """A native module that takes nothing."""

    def __getattr__(self, name):
        return lambda *args: None


def test_what_is_left_to_the_adapters():
    assert _cabi.load() is not None and _mix.load() is not None
    host, mix = _cabi._host, _mix._host
    x, w, s = torch.zeros(2, 128, dtype=BF16), torch.zeros(64, 128, dtype=torch.int8), torch.ones(64)
    sub = x.as_subclass(type("Sub", (torch.Tensor,), {}))
    for args in [(x, w, s, None), (x.cpu(), w, s, 3), (sub, w, s, None), (None, w, s, None), (x, w, s), (x, w, s, None, None)]:
        assert host.linear_int8(*args) is None
    assert host.linear_fp8(x, x, None, None, None, None, None, 0, None, 0, 0, 448.0, 1.0) is None
    assert host.linear_fp8(x, x, None, None, None, None, None, 1 << 70, None, 0, 0, 448.0, torch.ones(())) is None
    assert host.linear_fp8_backward(x, x, x, 1, None, None, None, None, 0, 1, 448.0, 1.0) is None
    assert host.quantize_block128_act(x) is None and host.mm_block128(x, x, s, s, None) is None
    assert host.attn_paged_decode(*[x] * 6, False, 1, 1.0) is None and host.attn_prefill(x, x, x, 0, 1.0) is None
    assert host.attn_paged_prefill(*[x] * 9, False, 1, True, 1.0) is None
    assert host.linear_fp8_operands(x, x, None, 1) is False and host.linear_fp8_operands(x, x, None, 2) is None
    assert mix.few_rows_linear(x, x, None, -1, 64, False) is None and mix.few_rows_linear_takes(sub, x, None, -1, 64) is None
    assert mix.sum_norm(x, None, True, 1e-5, None, None, None, None, 1.0, None) is None
    assert mix.residual_norm(x, x, s, s, 1.0, 1e-5) is None


def test_a_native_module_that_was_built_for_others_is_not_used(monkeypatch):
    from astrai_amd.extension import _native
    for adapter, name in ((_cabi, "_host"), (_mix, "_host_mix")):
        assert adapter.load() is not None
        module = adapter._host
        assert module.BUILT_FOR[:3] == (_native.CALLS_VERSION, adapter.ABI_VERSION, torch.__version__)
        older = [module.BUILT_FOR[:i] + ("older",) + module.BUILT_FOR[i + 1:] for i in range(4)]
        for built_for in (None, *older):
            with monkeypatch.context() as m:
                if built_for is None:   # not there at all
                    m.setitem(sys.modules, "astrai_amd.extension." + name, None)
                else:
                    m.setattr(module, "BUILT_FOR", built_for)
                m.setattr(adapter, "_lib", None)
                m.setattr(adapter, "_host", module)
                with pytest.warns(UserWarning, match=name + " is not used"):
                    assert adapter.load() is not None and adapter.load_error() is None   # the library is there all the same
                assert adapter._host.few_rows_parts(1) is None and adapter._host is not module


def test_nothing_is_taken_while_torch_traces():
    assert _cabi.load() is not None
    x, seen = torch.zeros(2, 128, dtype=BF16), []
    ask = lambda: seen.append(_cabi._host.linear_fp8_operands(x, x, None, 1))
    ask()
    torch.jit.trace(lambda t: (ask(), t + 1)[1], (x,), check_trace=False)
    ask()
    assert seen == [False, None, False]


def test_the_libraries_need_no_torch():
    """A machine without it builds the C ABI and leaves the native calls out."""
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "astrai_amd", "csrc")
    for target in ("all", "lib", "mix"):
        plan = subprocess.run(["make", "-n", "-B", "-C", csrc, "PYTHON=false", target], capture_output=True, text=True)
        assert plan.returncode == 0 and "libastrai_mix.so" in plan.stdout and "_host" not in plan.stdout, plan.stderr


def _rand(*shape, dtype=BF16, std=1.0):
    return (torch.randn(*shape, device="cuda") * std).to(dtype)


def _calls():
    """(call, whether the native form takes it) over the forms that operands come in."""
    def int8(k=512, n=384, **more):
        wq, sw = torch.randint(-127, 128, (n, k), device="cuda", dtype=torch.int8), torch.rand(n, device="cuda")
        return lambda x, bias=None: _cabi.linear_int8(x, wq, sw, bias)

    f = int8()
    yield lambda: f(_rand(3, 5, 512), _rand(384)), True
    yield lambda: f(_rand(512)), True
    yield lambda: f(_rand(512, 7).t()), False
    odd = int8(k=520)
    yield lambda: odd(_rand(9, 520)), False
    w, b, step = _rand(384, 512, std=0.02), _rand(384), torch.full((1,), 0.01, device="cuda")
    codes = w.float().div(0.01).to(torch.float8_e4m3fn)
    for x in (_rand(33, 512), _rand(2, 3, 512)):
        for c in (None, codes):
            yield lambda x=x, c=c: _cabi.linear_fp8(x, w, b, c, (None, step if c is not None else None), (None, None), 0, 448.0, 1.0), True

            def delayed(x=x, c=c):
                sx, sw, hx, hw = step.clone(), step.clone(), torch.ones(16, device="cuda"), torch.ones(16, device="cuda")
                out = _cabi.linear_fp8(x, w, None, c, (sx, sw), ((hx, 3), None if c is not None else (hw, 5)), 0, 448.0, 1.0)
                return out, sx, sw, hx, hw
            yield delayed, True
    sq, g = _rand(256, 256, std=0.02), _rand(48, 256)
    for want in (True, False):
        yield lambda want=want: _cabi.linear_fp8_backward(g, g, sq, want, None, None, 1, 57344.0, 1.0), True
    yield lambda: _cabi.quantize_fp8_block128_act(g), True
    yield lambda: _cabi.quantize_fp8_block128_act(_rand(256, 48).t()), False
    a8, sa = _cabi.quantize_fp8_block128_act(g)
    w8, sb = _cabi.quantize_fp8_block128_weight(_rand(200, 256))
    yield lambda: _cabi.mm_fp8_block128(a8, w8, sa, sb, _rand(200)), True
    yield lambda: _cabi.mm_fp8_block128(a8, w8, sa.t().contiguous().t(), sb), False
    for h, hkv, d in ((16, 4, 128), (8, 8, 64)):
        k, v, lens = _rand(500, hkv, d), _rand(500, hkv, d), [70, 1, 200]
        table = torch.randperm(500, device="cuda").int()[:450].reshape(3, 150).contiguous()
        table = torch.cat([table, table.flip(0)], 1).contiguous()
        rows, ind = torch.arange(3, device="cuda").int(), torch.tensor([0, 70, 71, 271], device="cuda").int()
        sched = _cabi.paged_prefill_schedule([40, 1, 130], "cuda")
        q1, qn = _rand(3, h, d), _rand(171, h, d)
        yield lambda q=q1, k=k, v=v, t=table: _cabi.attn_paged_decode(q, k, v, t, rows, ind), True
        yield lambda q=q1, k=k, v=v, t=table: _cabi.attn_paged_decode(q.flip(0).transpose(0, 1).contiguous().transpose(0, 1), k, v, t, rows, ind), False
        for c in (0, -1):
            yield lambda q=qn, k=k, v=v, t=table, c=c: _cabi.attn_paged_prefill(q, k, v, t, rows, ind, *sched, causal_offset=c), True
        x = _rand(2, 100, h + 2 * hkv, d)
        parts = x[:, :, :h], x[:, :, h:h + hkv], x[:, :, h + hkv:]
        yield lambda p=parts: _cabi.attn_prefill_qkv(*p, causal_offset=0, layout=1), True
        yield lambda p=parts: _cabi.attn_prefill_qkv(*(t.transpose(1, 2) for t in p), causal_offset=0, layout=0), False
    wide = _rand(20, 1024)
    yield lambda: _mix.few_rows_linear(wide[:, 256:768], w, b), True
    yield lambda: _mix.few_rows_linear(wide[:, 256:768], w, None, "silu"), True
    yield lambda: _mix.few_rows_linear(_rand(512), w, out_dtype=torch.float32), True
    vec, res = _rand(512, dtype=torch.float32), _rand(20, 512, dtype=torch.float32)
    yield lambda: _mix.sum_norm(wide[:, :512], vec, BF16, 1e-5, res, wide[:, 512:], vec, mult=0.5), True
    yield lambda: _mix.sum_norm(w, vec, BF16, 1e-5, tokens=torch.arange(20, device="cuda"), out=res.clone()), True
    yield lambda: _mix.residual_norm(_rand(20, 512), res.clone(), vec, vec, 0.5, 1e-5), True
    planes = _rand(3, 20, 512, dtype=torch.float32)
    yield lambda: _mix.few_rows_parts(wide[:, 256:768], w, 4), True
    yield lambda: _mix.few_rows_parts(_rand(2, 3, 512), w, 1), True
    yield lambda: _mix.sum_norm(planes, vec, BF16, 1e-5, res, res, vec, mult=0.5), True
    yield lambda: _mix.sum_norm(planes.repeat(1, 1, 2)[:, :, 512:], None, BF16, 1e-5), True
    yield lambda: _mix.residual_norm(planes, res.clone(), vec, vec, 0.5, 1e-5), True


@pytest.mark.gpu
def test_same_bits_as_the_adapters(monkeypatch):
    torch.manual_seed(3)
    calls = list(_calls())
    for i, (call, takes) in enumerate(calls):
        print("call", i, flush=True)
        torch.manual_seed(i)
        got = call()
        seen = []

        class Watched:
            def __init__(self, of):
                self.of = of

            def __getattr__(self, name):
                def run(*args):
                    seen.append((name, getattr(self.of, name)(*args)))
                    return seen[-1][1]
                return run

        with monkeypatch.context() as m:
            m.setattr(_cabi, "_host", Watched(_cabi._host))
            m.setattr(_mix, "_host", Watched(_mix._host))
            torch.manual_seed(i)
            call()
        assert any(r is not None for n, r in seen if n != "linear_fp8_operands") == takes, seen
        with monkeypatch.context() as m:
            m.setattr(_cabi, "_host", Refuses())
            m.setattr(_mix, "_host", Refuses())
            torch.manual_seed(i)
            want = call()
        for a, b in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
            assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.gpu
def test_errors_are_the_adapters():
    x, w = _rand(4, 256), _rand(64, 256)
    step = torch.ones(1, device="cuda")
    with pytest.raises(RuntimeError, match="inner dim mismatch"):
        _cabi.linear_fp8(x[:, :128].contiguous(), w, None, None, (None, None), (None, None), 0, 448.0, 1.0)
    with pytest.raises(RuntimeError, match="sx must be"):
        _cabi.linear_fp8(x, w, None, None, (step.double(), step), ((step, 0), (step, 0)), 0, 448.0, 1.0)
    with pytest.raises(RuntimeError, match="astrai_w8a8 error"):   # the library's own refusal, through the native call
        _cabi.linear_fp8(x, w, None, None, (step, step), ((step, 1), (step, 0)), 0, 448.0, 1.0)
    with pytest.raises(RuntimeError, match="multiple of 128"):
        _cabi.quantize_fp8_block128_act(_rand(4, 130))
    q, pool = _rand(2, 8, 128), _rand(64, 3, 128)
    ints = torch.zeros(2, 8, device="cuda").int(), torch.zeros(2, device="cuda").int(), torch.zeros(3, device="cuda").int()
    with pytest.raises(RuntimeError, match="divisible"):
        _cabi.attn_paged_decode(q, pool, pool, *ints)
    with pytest.raises(RuntimeError, match="not covered"):
        _mix.few_rows_linear(_rand(65, 256), w)


@pytest.mark.gpu
def test_both_forms_take_the_same_operands(monkeypatch):
    """The conditions stand in the native module and in the adapters: the same answers over every form of every operand."""
    def forms(rows, cols, dtype=BF16):
        t = _rand(rows * 2 + 1, cols * 2 + 16).to(dtype)
        yield t[:rows, :cols].contiguous()
        yield t[:rows, :cols]                                      # rows of a wider matrix
        yield t.flatten()[1:1 + rows * cols].view(rows, cols)      # at an odd address
        yield t.flatten()[4:4 + rows * cols].view(rows, cols)      # at 8 bytes
        yield t[:cols, :rows].t() if cols <= t.size(0) else t[:rows, 0:2 * cols:2]
        yield t[:rows, :cols].float()
        yield t[:rows, :cols].contiguous().cpu()
        yield t[:rows, :cols - 16].contiguous()
        yield t[:0, :cols]
        yield t[:rows, :cols].reshape(rows, 1, cols)

    def vectors(n):
        return [None, *(f.reshape(f.size(0), -1)[:, 0] if i == 4 else f.flatten() for i, f in enumerate(forms(1, n)) if i != 1)]

    asks = 0
    for x in (*forms(8, 256), *forms(65, 256), _rand(256)):
        for w in forms(64, 256):
            if w.dim() != 2:
                continue
            for bias in vectors(64):
                calls = [lambda: _cabi.linear_fp8_operands(x, w, bias), lambda: _cabi.linear_fp8_operands(x, w, bias, 0)]
                calls += [lambda act=act: _mix.few_rows_linear_supported(x, w, bias, act) for act in (None, "silu")]
                for call in calls:
                    with monkeypatch.context() as m:
                        m.setattr(_cabi, "_host", Refuses())
                        m.setattr(_mix, "_host", Refuses())
                        want = call()
                    assert call() == want, (x.shape, x.stride(), x.dtype, w.shape, w.stride(), w.dtype, bias is None or bias.shape)
                    asks += 1
    assert asks > 5000
