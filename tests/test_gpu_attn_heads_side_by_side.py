"""Paged steps of the general kernel, whose waves take KV heads side by side where a split's share of the slot table is 120
positions or more and splits side by side otherwise: both sides of that line, KV heads that fill no whole workgroup."""

import pytest
import torch

from oracle import decoder_oracle as D
from tests.helpers import assert_bf16_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("h,hkv,d", [(6, 3, 64), (5, 5, 32), (16, 16, 64), (7, 1, 256)])
@pytest.mark.parametrize("width,nsplit", [(119, 1), (120, 1), (720, 2), (720, 5), (720, 6), (719, 6), (720, 7), (7680, 64), (7679, 64)])
def test_either_order(h, hkv, d, width, nsplit):
    from astrai_amd.extension import _cabi
    print(f"case h={h} hkv={hkv} d={d} width={width} nsplit={nsplit}", flush=True)
    g = torch.Generator().manual_seed(width + nsplit + h)
    lens = [min(width, n) for n in (width, 1, 117, 0, 720)]
    pool = sum(lens) + 3
    q, k, v = (torch.randn(n, heads, d, generator=g).to(torch.bfloat16) for n, heads in ((len(lens), h), (pool, hkv), (pool, hkv)))
    slots, table, at = torch.randperm(pool, generator=g).int(), torch.full((len(lens), width), -1, dtype=torch.int32), 0
    for i, n in enumerate(lens):
        table[i, :n] = slots[at:at + n]
        at += n
    rows = torch.arange(len(lens), dtype=torch.int32)
    indptr = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    args = (q, k, v, table, rows, indptr)
    got = _cabi.attn_paged_decode(*(t.to(DEV) for t in args), nsplit=nsplit)
    assert_bf16_close(got, D.attn_paged_decode(*args), what=f"{nsplit} splits of {width}")


def test_splits_of_uneven_pairs():
    from astrai_amd.extension import _cabi
    rows, tuned = _cabi._rows_decode_nsplit, _cabi.paged_nsplit
    assert [rows(p, w) for p, w in ((1536, 479), (1600, 479), (1600, 480), (1792, 8192), (2048, 8192), (2049, 8192))] == [2, 1, 2, 1, 1, 1]
    assert [tuned(p, w) for p, w in ((256, 8192), (320, 799), (320, 800), (568, 799), (568, 800), (512, 8192), (500, 8192), (2049, 8192))] == \
        [3, 2, 3, 1, 3, 1, 1, 1]


@pytest.mark.parametrize("b,h,hkv,d", [(41, 8, 8, 128), (71, 32, 8, 128), (201, 16, 8, 64)])
def test_steps_with_splits_of_uneven_pairs(b, h, hkv, d):
    from astrai_amd.extension import _cabi
    g = torch.Generator(device=DEV).manual_seed(b)
    width, pool = 816, 1200
    print(f"case b={b} h={h} hkv={hkv} d={d}", flush=True)
    q, k, v = (torch.randn(n, heads, d, generator=g, device=DEV).to(torch.bfloat16) for n, heads in ((b, h), (pool, hkv), (pool, hkv)))
    table = torch.randint(0, pool, (b, width), generator=g, device=DEV, dtype=torch.int32)
    lens = torch.randint(1, width + 1, (b,), generator=g, device=DEV)
    lens[:3] = torch.tensor([1, width, 16], device=DEV)
    rows = torch.arange(b, device=DEV, dtype=torch.int32)
    indptr = torch.cat([lens.new_zeros(1), lens.cumsum(0)]).int()
    args = (q, k, v, table, rows, indptr)
    assert (_cabi._rows_decode_nsplit if d == 64 else _cabi.paged_nsplit)(b * hkv, width) == (2 if d == 64 else 3)
    assert_bf16_close(_cabi.attn_paged_decode(*args), D.attn_paged_decode(*(t.cpu() for t in args)), what=f"{b} x {hkv} pairs")
