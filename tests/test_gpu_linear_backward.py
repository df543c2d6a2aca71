"""The bf16 backward of a Linear on its own kernels, against 64-bit products of the same operands."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operands(m, n, k, seed=0):
    r = torch.Generator().manual_seed(seed + m * 7 + n * 3 + k)
    return (torch.randn(m, n, generator=r).mul(0.01).bfloat16().to(DEV), torch.randn(m, k, generator=r).bfloat16().to(DEV),
            torch.randn(n, k, generator=r).mul(0.02).bfloat16().to(DEV))


def _check(got, a, b, what):
    """One rounding to bf16 (2^-9 of the value, twice that for the rounding of what the fp32 sums are off), and fp32 sums of
    t terms, each within 2^-24 of the partial sums, which the terms' magnitudes bound."""
    a, b = a.double(), b.double()
    want, bound = a @ b, a.abs() @ b.abs()
    bad = (got.double() - want).abs() > want.abs() * 2.0 ** -8 + bound * (a.size(1) * 2.0 ** -24)
    assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.numel()} outside"


# tiles are 128 x 128, slabs 64 deep through rings of four and of two stages; contractions in one range and in several
@pytest.mark.parametrize("m,n,k", [(1, 64, 8), (3, 128, 128), (63, 64, 120), (64, 192, 136), (65, 256, 1000), (127, 320, 264),
                                   (129, 384, 128), (256, 448, 2048), (300, 3072, 2048), (37, 4096, 1024), (552, 11264, 512),
                                   (5000, 64, 72), (1700, 2048, 2048), (700, 2048, 5632), (200, 2112, 4104)])
def test_gradients(m, n, k):
    from astrai_amd.extension import _cabi
    print(f"case m={m} n={n} k={k}", flush=True)
    g, x, w = _operands(m, n, k)
    gx, gw, gb = _cabi.linear_backward(g, x, w, (True, True, True))
    _check(gx, g, w, "input")
    _check(gw, g.t(), x, "weight")
    _check(gb[None], torch.ones(1, m, device=DEV), g, "bias")
    again = _cabi.linear_backward(g, x, w, (True, True, True))
    assert all(torch.equal(a, b) for a, b in zip((gx, gw, gb), again))
    # each by itself is the same
    assert torch.equal(_cabi.linear_backward(g, x, w, (True, False, False))[0], gx)
    ax, aw, ab = _cabi.linear_backward(g, x, w, (False, True, False))
    assert torch.equal(aw, gw) and ax.numel() == 0 and ab.numel() == 0


@pytest.mark.parametrize("m,n,k", [(700, 128, 5632), (2200, 320, 2056)])
def test_input_gradient_of_more_than_a_round(m, n, k):
    """Through the C entry, which takes what the adapter leaves to the library: two workgroups to a compute unit."""
    from astrai_amd.extension import _cabi
    print(f"case m={m} n={n} k={k}", flush=True)
    lib = _cabi.load()
    g, x, w = _operands(m, n, k)
    out = torch.full((m + 8, k), -777.0, device=DEV, dtype=torch.bfloat16)
    scratch = torch.empty(max(1, lib.astrai_w8a8_linear_backward_scratch_bytes(m, n, k)), device=DEV, dtype=torch.uint8)
    assert lib.astrai_w8a8_linear_backward_bf16(g.data_ptr(), x.data_ptr(), w.data_ptr(), scratch.data_ptr(), out.data_ptr(), None, None,
                                                m, n, k, torch.cuda.current_stream().cuda_stream) == 0
    _check(out[:m], g, w, "input")
    assert torch.all(out[m:] == -777.0), "rows past M were written"


def test_what_is_not_finite_stays_in_its_row_or_column():
    from astrai_amd.extension import _cabi
    g, x, w = _operands(200, 192, 200)
    g[5, 7], x[3, 199], w[11, 0] = float("nan"), float("inf"), float("-inf")
    gx, gw, gb = _cabi.linear_backward(g, x, w, (True, True, True))
    want = (g.float() @ w.float(), g.float().t() @ x.float(), g.float().sum(0))
    for a, b in zip((gx, gw, gb), want):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())


@pytest.mark.parametrize("shape,n", [((2, 150, 256), 640), ((300, 256), 320)])
def test_autograd_takes_it(shape, n):
    """F.linear's gradients with no policy on, leading dimensions and all; what the kernels do not take goes the plain way."""
    import torch.nn.functional as F
    import astrai_amd.extension.fp8  # noqa: F401  (installs the hook)
    k = shape[-1]
    r = torch.Generator().manual_seed(n)
    x = torch.randn(*shape, generator=r).bfloat16().to(DEV).requires_grad_(True)
    w = torch.randn(n, k, generator=r).mul(0.05).bfloat16().to(DEV).requires_grad_(True)
    b = torch.zeros(n, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    for dense in (True, False):
        g = torch.randn(*shape[:-1], n, generator=r).bfloat16().to(DEV)
        if not dense:
            g = g[..., :1].expand(*shape[:-1], n)
        gx, gw, gb = torch.autograd.grad(F.linear(x, w, b), (x, w, b), g)
        assert gx.shape == x.shape
        g2, x2 = g.reshape(-1, n), x.detach().reshape(-1, k)
        _check(gx.reshape(-1, k), g2, w.detach(), "input")
        _check(gw, g2.t(), x2, "weight")
        _check(gb[None], torch.ones(1, g2.size(0), device=DEV), g2, "bias")


def test_replayed_graph():
    """Contractions in several ranges, with their planes, in a captured graph."""
    from astrai_amd.extension import _cabi
    g, x, w = _operands(300, 4096, 1024)
    _cabi.linear_backward(g, x, w, (True, True, True))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _cabi.linear_backward(g, x, w, (True, True, True))
    for seed in range(3):
        for t, new in zip((g, x, w), _operands(300, 4096, 1024, seed)):
            t.copy_(new)
        graph.replay()
        torch.cuda.synchronize()
        want = _cabi.linear_backward(g, x, w, (True, True, True))
        assert all(torch.equal(a, b) for a, b in zip(out, want))
