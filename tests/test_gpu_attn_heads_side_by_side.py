"""Paged steps of the general kernel, whose waves take KV heads side by side where the slot table has 480 positions or
more and a split's share of them is 120, and splits side by side otherwise: both sides of those lines, KV heads that fill no whole
workgroup."""

import pytest
import torch

from oracle import decoder_oracle as D
from tests.helpers import assert_bf16_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("h,hkv,d", [(6, 3, 64), (5, 5, 32), (16, 16, 64), (7, 1, 256)])
@pytest.mark.parametrize("width,nsplit", [(119, 1), (120, 1), (479, 2), (480, 2), (480, 4), (480, 5), (720, 2), (720, 5), (720, 6), (719, 6), (720, 7), (7680, 64), (7679, 64)])
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


def test_splits_are_no_more_behind_a_wide_table():
    """The table's width says nothing of the contexts: 100 keys each of 100 sequences, 16 KV heads, took twice the time in three splits."""
    from astrai_amd.extension import _cabi
    assert [_cabi.paged_nsplit(p, 8192) for p in (257, 320, 384, 385, 568, 1600, 2048)] == [2, 2, 2, 1, 1, 1, 1]
    assert [_cabi._rows_decode_nsplit(p, 8192) for p in (1536, 1537, 1600, 2048)] == [2, 1, 1, 1]


@pytest.mark.parametrize("b,h,hkv,d", [(41, 8, 8, 128), (71, 32, 8, 128), (201, 16, 8, 64)])
def test_steps_of_uneven_pairs(b, h, hkv, d):
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
    want = D.attn_paged_decode(*(t.cpu() for t in args))
    for nsplit in (0, 2, 3):
        assert_bf16_close(_cabi.attn_paged_decode(*args, nsplit=nsplit), want, what=f"{b} x {hkv} pairs, {nsplit} splits")
