"""128-block scaled products whose steps arrive four slabs at a time: every count of slabs modulo four, ragged rows and
columns, in the kernels of 64 x 64, 128 x 128 and 256 x 256 tiles."""

import pytest
import torch

from oracle import w8a8_oracle as O
from tests.helpers import assert_bf16_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (5 slabs are the fewest of the 128 x 128 tiles' ring of four stages, one and four those of its two stages)
@pytest.mark.parametrize("m,n,slabs,kernel", [(65 + 7 * s, 200 if s % 2 else 333, s, "small64") for s in range(1, 10)] +
                         [(1100, 2048, s, "mid128_block128") for s in (1, 4, 5, 6, 7, 8, 9)] + [(1301, 1804, 11, "mid128_block128"), (1100, 2045, 6, "mid128_block128"), (1029, 2047, 4, "mid128_block128")] +
                         [(2500, 4096, s, "pingpong_block128") for s in (2, 3, 4, 5, 6, 9)])
def test_steps_of_every_slab(m, n, slabs, kernel):
    """Steps spread over seven octaves from row to row and from block to block: one of another row, column block or slab
    changes results by factors."""
    from astrai_amd.extension import _cabi
    from astrai_amd.extension.ops import fp8_block as blk
    print(f"case m={m} n={n} slabs={slabs}", flush=True)
    g = torch.Generator().manual_seed(slabs * 1000 + m)
    k = 128 * slabs
    a8 = torch.randn(m, k, generator=g).to(torch.float8_e4m3fn)
    b8 = torch.randn(n, k, generator=g).to(torch.float8_e4m3fn)
    sa = 2.0 ** (torch.rand(m, slabs, generator=g) * 7 - 5)
    sb = 2.0 ** (torch.rand((n + 127) // 128, slabs, generator=g) * 7 - 5)
    out = blk.mm_fp8_blockscaled(a8.to(DEV), b8.to(DEV), sa.to(DEV), sb.to(DEV))
    assert _cabi.last_kernel() == kernel
    assert_bf16_close(out, O.fp8_gemm_blockscaled(a8, b8, sa, sb), what=f"{kernel} of {slabs} slabs")
