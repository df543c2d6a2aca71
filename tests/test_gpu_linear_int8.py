"""The int8 Linear as one library call, against its two steps: operands as the kernels take them, and those that go the long
way (strides, inner sizes off the vector grid, strided steps and biases), bit for bit; refused operands stay refused."""
import pytest
import torch
import torch.nn.functional as F

from astrai_amd.extension import _cabi, w8a8

pytestmark = pytest.mark.gpu


def data(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16().cuda()


def steps(x, wq, sw, bias):
    xq, sx = _cabi.quantize_int8_rows(x)
    return _cabi.mm_int8(xq, wq, sx, sw, bias).reshape(*x.shape[:-1], wq.size(0))


@pytest.mark.parametrize("rows", [(1,), (16,), (3, 43), (129,), (2, 700), (1, 1, 5)], ids=str)
@pytest.mark.parametrize("k,n", [(16, 8), (48, 40), (2048, 3072), (130, 24), (1000, 7), (32, 1)])
def test_one_call_is_the_two_steps(rows, k, n):
    print("linear int8", rows, k, n, flush=True)
    wq, sw = _cabi.quantize_int8_rows(data(1, n, k))
    sw, bias = sw.reshape(-1), data(2, n)
    x = data(3, *rows, k)
    wide = data(4, *rows, 2 * k)[..., ::2]
    for inp in (x, wide, x[..., :], x.transpose(0, 1) if x.dim() > 2 else x):
        for b in (None, bias, data(5, n, 2)[:, 0]):
            got = _cabi.linear_int8(inp, wq, sw, b)
            assert got.shape == (*inp.shape[:-1], n) and torch.equal(got, steps(inp, wq, sw, b))
    assert torch.equal(_cabi.linear_int8(x[(0,) * (x.dim() - 1)], wq, sw), steps(x, wq, sw, None).reshape(-1, n)[0])
    assert torch.equal(_cabi.linear_int8(x, wq.t().contiguous().t(), sw.repeat_interleave(2)[::2], bias), steps(x, wq, sw, bias))


def test_refused_operands():
    x, (wq, sw) = data(1, 4, 64), _cabi.quantize_int8_rows(data(2, 8, 64))
    sw = sw.reshape(-1)
    for bad in ((x.float(), wq, sw, None), (x, wq.float(), sw, None), (x, wq, sw[:7], None), (x, wq, sw.half(), None),
                (x, wq, sw, sw), (x, wq[:, :48], sw, None), (x.cpu(), wq, sw, None), (x, wq.cpu(), sw, None),
                (x.reshape(-1)[1:65].reshape(1, 64), wq, sw, None)):
        with pytest.raises((RuntimeError, TypeError)):
            _cabi.linear_int8(*bad)


def test_through_the_linear_hook_eager_captured_and_with_gradients():
    x, w, b = data(1, 16, 512), data(2, 256, 512), data(3, 256)
    wq, sw = _cabi.quantize_int8_rows(w)
    want = steps(x, wq, sw.reshape(-1), b)
    with w8a8.int8_autocast():
        with torch.no_grad():
            assert torch.equal(F.linear(x, w, b), want)
            graph, held = torch.cuda.CUDAGraph(), x.clone()
            with torch.cuda.graph(graph):
                out = F.linear(held, w, b)
            for seed in (4, 5):
                held.copy_(data(seed, 16, 512))
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(out, steps(held, wq, sw.reshape(-1), b))
        leaf = x.clone().requires_grad_()
        y = F.linear(leaf, w, b)
        y.float().sum().backward()
        assert torch.equal(y.detach(), want) and leaf.grad.shape == x.shape and bool(leaf.grad.isfinite().all())
        # batching takes the Linear apart above the hook: the bf16 product, then the bias, one rounding each
        rows = torch.func.vmap(lambda t: F.linear(t, w, b))(x)
        prod, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        bound = 2.0 ** -8 * (prod.abs() + (prod + b.double()).abs()) * 1.01 + 512 * 2.0 ** -24 * size
        assert bool(((rows.double() - prod - b.double()).abs() <= bound).all())
