"""The fp8 backward of a Linear over token counts that no product takes whole: the transposed codes are padded with zeros,
the bias gradient is summed where the gradient is quantized. Against the decoded codes in 64 bits."""
import pytest
import torch

from astrai_amd.extension import _cabi
from helpers import assert_bf16_close

pytestmark = pytest.mark.gpu


def operands(m, k, seed):
    g = torch.Generator().manual_seed(seed)
    return [(torch.randn(*s, generator=g) * std).bfloat16().cuda() for s, std in (((m, k), 0.01), ((m, k), 1.0), ((k, k), 1.0))]


@pytest.mark.parametrize("masks", [(True, True, True), (False, True, True), (True, True, False), (False, True, False)], ids=str)
@pytest.mark.parametrize("m,k", [(1, 128), (16, 256), (17, 256), (112, 128), (127, 256), (128, 128), (129, 200), (1001, 256),
                                 (2064, 384), (333, 1000), (5, 100)])
def test_ragged_tokens(m, k, masks):
    print("ragged backward", m, k, masks, flush=True)
    g, x, w = operands(m, k, m)
    for fmt, top in ((1, 57344.0), (0, 448.0)):
        steps = [(t.float().abs().max() / lim).reshape(1) for t, lim in ((g, top), (w, top), (x, top))]
        gx, gw, gb, amax = _cabi.linear_backward_fp8(g, x, w, masks, *steps, fmt)
        dec = [_cabi.quantize_bf16(t, s, fmt)[0].double() * s.double() for t, s in ((g, steps[0]), (w, steps[1]), (x, steps[2]))]
        # (the bound by which the fp8 products are compared with the oracle everywhere: the matrix instruction aligns
        # the products of a step before it adds them, padded or not)
        assert_bf16_close(gw.cpu(), (dec[0].T @ dec[2]).cpu(), what="weight gradient")
        if masks[0]:
            assert_bf16_close(gx.cpu(), (dec[0] @ dec[1]).cpu(), what="input gradient")
            assert float(amax) == float(g.float().abs().max())
        if masks[2]:   # fp32: at most m roundings of the sum of magnitudes, then one to bf16
            want, size = g.double().sum(0), g.double().abs().sum(0)
            assert gb.dtype == torch.bfloat16 and gb.shape == (k,)
            assert bool(((gb.double() - want).abs() <= 2.0 ** -8 * want.abs() + m * 2.0 ** -24 * size).all())


def test_padding_is_zeros_and_nothing_else_moves():
    for m, k, fmt in ((100, 72, 0), (1001, 264, 1), (130, 13, 0)):
        g = operands(m, k, 5)[0]
        step = torch.full((1,), 0.001, device="cuda")
        ldt = -(-m // 128) * 128
        x8, x8t = _cabi._quantize_transposed(g, step, fmt, ldt, True)
        want, want_t, _ = _cabi.quantize_transpose_bf16(g, step, fmt, want_rowmajor=True)
        assert torch.equal(x8.view(torch.uint8), want.view(torch.uint8))
        assert torch.equal(x8t[:, :m].view(torch.uint8), want_t.view(torch.uint8))
        assert not x8t[:, m:].view(torch.uint8).any()


def test_infinities_and_nans_reach_the_sums():
    g, x, w = operands(300, 128, 9)
    g[7, 3], g[200, 9] = float("inf"), float("nan")
    step = torch.ones(1, device="cuda")
    _, _, gb, amax = _cabi.linear_backward_fp8(g, x, w, (True, True, True), step, step, step, 1)
    assert float(gb[3]) == float("inf") and bool(gb[9].isnan()) and float(amax) == float("inf")
    assert bool(gb[torch.tensor([i not in (3, 9) for i in range(128)], device="cuda")].isfinite().all())


@pytest.mark.parametrize("masks", [(True, True, True), (True, True, False), (False, True, True)], ids=str)
def test_no_tokens(masks):
    g, x, w = operands(0, 128, 1)
    step = torch.ones(1, device="cuda")
    gx, gw, gb, amax = _cabi.linear_backward_fp8(g, x, w, masks, step, step, step, 1)
    assert gx.shape == x.shape and not gw.any() and float(amax) == 0.0
    assert not masks[2] or (gb.shape == (128,) and not gb.any())
