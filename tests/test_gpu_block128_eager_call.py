"""The block-scaled product's direct call: taken for plain eager operands alone, with the op's bits; what stands above a device
kernel (modes, transforms, traces, gradients) sees the op."""

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

DEV = "cuda"


def _operands(m=9, n=200, k=256, device=DEV):
    r = torch.Generator().manual_seed(4)
    a8, b8 = (torch.randn(rows, k, generator=r).to(torch.float8_e4m3fn).to(device) for rows in (m, n))
    return a8, b8, torch.rand(m, k // 128, generator=r).to(device), torch.rand((n + 127) // 128, k // 128, generator=r).to(device)


def test_operands_off_the_gpu_reach_the_op():
    from astrai_amd.extension.ops import fp8_block as blk
    with pytest.raises(RuntimeError, match="no CPU implementation"):
        blk.mm_fp8_blockscaled(*_operands(device="cpu"))


@pytest.mark.gpu
def test_plain_operands_take_the_direct_call(monkeypatch):
    from astrai_amd.extension import _cabi
    from astrai_amd.extension.ops import fp8_block as blk
    args = _operands()
    want = torch.ops.custom.fp8_gemm_blockscaled(*args)
    with monkeypatch.context() as m:
        m.setattr(blk, "fp8_gemm_blockscaled", None)   # (not called)
        got = blk.mm_fp8_blockscaled(*args)
        with torch.no_grad(), torch.autocast("cuda", torch.bfloat16):
            again = blk.mm_fp8_blockscaled(*args, None)
    assert torch.equal(got, want) and torch.equal(again, want) and got.dtype == torch.bfloat16
    assert _cabi.mm_fp8_block128_eager(args[0].t().contiguous().t(), *args[1:]) is None   # left to the op, which copies
    assert torch.equal(blk.mm_fp8_blockscaled(args[0].t().contiguous().t(), *args[1:]), want)


@pytest.mark.gpu
def test_what_stands_above_sees_the_op():
    from astrai_amd.extension import _cabi
    from astrai_amd.extension.ops import fp8_block as blk
    args = _operands()
    want = blk.mm_fp8_blockscaled(*args)
    direct = lambda *a: _cabi.mm_fp8_block128_eager(*(a or args))  # noqa: E731
    assert direct() is not None
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, rest=(), kwargs=None):
            seen.append(str(func))
            return func(*rest, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, rest=(), kwargs=None):
            return func(*rest, **(kwargs or {}))

    with Dispatch():
        assert direct() is None
        assert torch.equal(blk.mm_fp8_blockscaled(*args), want)
    assert any("fp8_gemm_blockscaled" in s for s in seen)
    with Function():
        assert direct() is None
        assert torch.equal(blk.mm_fp8_blockscaled(*args), want)
    taken = []
    step = args[2].clone().requires_grad_(True)
    assert direct(*args[:2], step, args[3]) is None
    with torch.no_grad():
        assert direct(*args[:2], step, args[3]) is not None
    torch.func.vmap(lambda t: (taken.append(direct(*args[:2], t, args[3])), t)[1])(torch.stack([args[2]] * 2))
    torch.func.vmap(lambda t: (taken.append(direct()), t)[1])(torch.zeros(2, device=DEV))
    torch.func.grad(lambda t: (taken.append(direct(*args[:2], t, args[3])), t.sum())[1])(args[2])
    torch.func.functionalize(lambda t: (taken.append(direct(*args[:2], t, args[3])), t)[1])(args[2])
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(args[2], torch.ones_like(args[2]))
        taken.append(direct(*args[:2], dual, args[3]))
    torch.jit.trace(lambda t: (taken.append(direct()), t + 1)[1], (step.detach(),), check_trace=False)
    taken.append(direct(*args[:2], args[2].as_subclass(type("Sub", (torch.Tensor,), {})), args[3]))
    assert taken == [None] * 7


@pytest.mark.gpu
def test_a_profile_has_the_op():
    from torch.profiler import ProfilerActivity, profile
    from astrai_amd.extension import _cabi
    from astrai_amd.extension.ops import fp8_block as blk
    args = _operands()
    want = blk.mm_fp8_blockscaled(*args)
    with profile(activities=[ProfilerActivity.CPU]) as p:
        assert _cabi.mm_fp8_block128_eager(*args) is None
        got = blk.mm_fp8_blockscaled(*args)
    assert torch.equal(got, want) and any("fp8_gemm_blockscaled" in e.key for e in p.key_averages())
    assert _cabi.mm_fp8_block128_eager(*args) is not None


@pytest.mark.gpu
def test_bf16_backward_native_and_adapter(monkeypatch):
    """The native form of the bf16 backward and the adapter's own path: the same bits, the same refusals."""
    from astrai_amd.extension import _cabi

    class Refuses:
        def __getattr__(self, name):
            return lambda *args: None

    r = torch.Generator().manual_seed(2)
    mk = lambda *s: torch.randn(*s, generator=r).bfloat16().to(DEV)  # noqa: E731
    g, x, w = mk(70, 192), mk(70, 136), mk(192, 136)
    forms = [(g, x, w), (g[:, :128].contiguous(), x, w[:128]), (g.t().contiguous().t(), x, w), (g, x[:, 8:], w[:, 8:].contiguous()),
             (g, x.float(), w), (g[:, :100].contiguous(), x, w[:100].contiguous()), (g, x[:69], w), (g[:0], x[:0], w),
             (g, x, w.flatten()[1:1 + 191 * 136].view(191, 136)), (g, x[:, :130].contiguous(), w[:, :130].contiguous())]
    for i, (a, b, c) in enumerate(forms):
        for masks in ((True, True, True), (False, True, False), (True, False, False), (False, False, True), (False, False, False)):
            got = _cabi.linear_backward(a, b, c, masks)
            with monkeypatch.context() as m:
                m.setattr(_cabi, "_host", Refuses())
                want = _cabi.linear_backward(a, b, c, masks)
            assert (got is None) == (want is None), (i, masks)
            if got is not None:
                assert all(p.shape == q.shape and torch.equal(p, q) for p, q in zip(got, want)), (i, masks)
    assert _cabi.linear_backward(*forms[0], (True, True, True)) is not None and _cabi._host.linear_backward(g, x, w, True, True, True)
