"""8-bit products on tiles of 128 x 256, of 128 x 128 and, one to a compute unit, of 64 x 64: every remainder of rows, columns and slabs, and columns whose rows of
outputs are whole 16-byte pieces, whole 8-byte pieces or neither."""

import pytest
import torch

from tests.helpers import assert_bf16_close

pytestmark = pytest.mark.gpu
DEV = "cuda"

# rows, columns, K, kernel: 1 to 7 slabs (three stages, two slabs a turn); one row or column past a tile, one short of it
CASES = [(2049, 2049, 128, "mid128x256"), (2047, 2302, 256, "mid128x256"), (2100, 2060, 384, "mid128x256"), (1281, 3080, 512, "mid128x256"),
         (4090, 1100, 640, "mid128x256"), (300, 11264, 768, "mid128x256"), (129, 16640, 896, "mid128x256"), (16512, 256, 640, "mid128x256"),
         (1500, 1501, 128, "mid128"), (1530, 1500, 640, "mid128"), (1409, 1544, 768, "mid128"), (1537, 1410, 384, "mid128")] + [
    # one group of waves up to nine slabs (eleven with one step), then halves of K: odd and even counts of slabs
    (130 + 9 * i, 1021 + i, 128 * i, "small64") for i in (1, 2, 3, 4, 5, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17)]


@pytest.mark.parametrize("m,n,k,kernel", CASES)
def test_int8(m, n, k, kernel):
    from astrai_amd.extension import _cabi
    print(f"case m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = torch.randint(-128, 128, (m, k), generator=g, device=DEV, dtype=torch.int8)
    b = torch.randint(-128, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
    sa, sb = (torch.rand(i, generator=g, device=DEV) + 0.5 for i in (m, n))
    bias = (torch.randn(n, generator=g, device=DEV) * k).to(torch.bfloat16)
    out = _cabi.mm_int8(a, b, sa, sb, bias)
    assert _cabi.last_kernel() == kernel
    acc = (a.double() @ b.double().t()).float()   # whole numbers below 2^24
    assert torch.equal(out, (acc * sa[:, None] * sb + bias.float()).to(torch.bfloat16))
    assert torch.equal(_cabi.mm_int8(a, b, sa, sb), (acc * sa[:, None] * sb).to(torch.bfloat16))


@pytest.mark.parametrize("m,n,k,kernel", CASES)
@pytest.mark.parametrize("fmt", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_fp8(m, n, k, kernel, fmt):
    from astrai_amd.extension import _cabi
    print(f"case m={m} n={n} k={k} {fmt}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a, b = (torch.randn(i, k, generator=g, device=DEV).to(fmt) for i in (m, n))
    bias = torch.randn(n, generator=g, device=DEV).to(torch.bfloat16)
    acc, one, half = a.double() @ b.double().t(), torch.ones(1, device=DEV), torch.full((1,), 0.5, device=DEV)
    out = _cabi.mm_fp8(a, b, one, half, 0, None, bias)
    assert _cabi.last_kernel() == kernel
    assert_bf16_close(out, (acc * 0.5 + bias.double()).to(torch.bfloat16), what="one step")
    out = _cabi.mm_fp8(a, b, one, half, 0, None, bias, True)
    assert torch.equal(out, _cabi.mm_fp8(a, b, one, half) + bias)
    sa, sb = (torch.rand(i, generator=g, device=DEV) + 0.5 for i in (m, n))
    out = _cabi.mm_fp8(a, b, sa, sb, 0, None, bias)
    exact = acc * sa[:, None].double() * sb.double() + bias.double()
    assert_bf16_close(out, exact.to(torch.bfloat16), what="a step per row and column")


@pytest.mark.parametrize("slabs", [40, 41, 42, 43, 45, 46])
def test_block128_in_two_halves(slabs):
    """Steps spread over seven octaves; a row's step that is not a number stays in its row, also where the second half of the row
    ahead of it is a slab short."""
    from astrai_amd.extension import _cabi
    from oracle import w8a8_oracle as O
    m, n, k = 70 + slabs, 200, 128 * slabs
    print(f"case m={m} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(slabs)
    a, b = (torch.randn(i, k, generator=g).to(torch.float8_e4m3fn) for i in (m, n))
    sa = 2.0 ** (torch.rand(m, slabs, generator=g) * 7 - 5)
    sb = 2.0 ** (torch.rand((n + 127) // 128, slabs, generator=g) * 7 - 5)
    want = O.fp8_gemm_blockscaled(a, b, sa, sb)
    out = _cabi.mm_fp8_block128(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV))
    assert _cabi.last_kernel() == "small64"
    assert_bf16_close(out, want, what=f"{slabs} slabs")
    sa[5, 0], sb[1, 0] = float("nan"), float("inf")
    out = _cabi.mm_fp8_block128(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV)).cpu()
    assert out[5].isnan().all() and torch.isfinite(out[torch.arange(m) != 5, :128]).all()
    assert not torch.isfinite(out[:, 128:]).any()


@pytest.mark.parametrize("slabs,n", [(2, 3716), (3, 3713), (4, 3712), (5, 3716), (6, 3716), (7, 3716), (8, 3716), (9, 3715), (10, 3712), (11, 3716), (12, 3720), (13, 3713), (14, 3584)])
def test_block128_wide(slabs, n):
    """Every count of slabs modulo four (steps come four at a time) and three (stages); steps spread over seven octaves, one of them
    not a number."""
    from astrai_amd.extension import _cabi
    from oracle import w8a8_oracle as O
    m, k = 1163, 128 * slabs
    print(f"case m={m} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(slabs)
    a, b = (torch.randn(i, k, generator=g).to(torch.float8_e4m3fn) for i in (m, n))
    sa = 2.0 ** (torch.rand(m, slabs, generator=g) * 7 - 5)
    sb = 2.0 ** (torch.rand((n + 127) // 128, slabs, generator=g) * 7 - 5)
    want = O.fp8_gemm_blockscaled(a, b, sa, sb)
    run = lambda: _cabi.mm_fp8_block128(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV))   # noqa: E731
    out = run()
    assert _cabi.last_kernel() == "mid128x256_block128"
    assert_bf16_close(out, want, what=f"{slabs} slabs")
    sa[5, slabs // 2], sb[3, slabs - 1] = float("nan"), float("inf")
    out, hit = run().cpu(), torch.zeros(m, n, dtype=torch.bool)
    hit[5], hit[:, 384:512] = True, True
    assert torch.equal(~torch.isfinite(out), hit)
