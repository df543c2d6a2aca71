"""Merging of context splits: split counts on both sides of the groups a workgroup has, head counts that no power of two
divides, sequences shorter than their splits, and the calls that merge nothing. Against the same call with one split."""
import pytest
import torch

from astrai_amd.extension import _cabi

pytestmark = pytest.mark.gpu


def close(got, want, v):
    # Both are bf16 roundings (2^-8 each) of the same sum: probabilities add up to 1, a context of at most 2048 keys is
    # summed in fp32, 2^-24 a key of at most max |v|.
    bound = 2.0 ** -7 * want.double().abs() + 2048 * 2.0 ** -24 * v.double().abs().max()
    assert bool(((got.double() - want.double()).abs() <= bound).all())


@pytest.mark.parametrize("h,hkv,d", [(16, 4, 128), (6, 2, 128), (8, 1, 128), (40, 8, 128), (32, 8, 64), (9, 3, 64), (5, 5, 32), (12, 4, 256)])
def test_paged_splits(h, hkv, d):
    g = torch.Generator().manual_seed(h * d)
    kv = [1, 700, 63, 64, 2048, 17]
    b, slots = len(kv), sum(kv)
    q, k, v = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((b, h, d), (slots, hkv, d), (slots, hkv, d)))
    table, at = torch.full((b, 2100), -1, dtype=torch.int32), 0
    for i, n in enumerate(kv):
        table[i, :n] = torch.arange(at, at + n)
        at += n
    rows, ind = torch.arange(b, dtype=torch.int32).cuda(), torch.tensor([0] + kv).cumsum(0).int().cuda()
    table = table.cuda()
    one = _cabi.attn_paged_decode(q, k, v, table, rows, ind, nsplit=1)
    spot = torch.softmax((q[4].double().reshape(hkv, h // hkv, d) * d ** -0.5)
                         @ k[828:2876].double().permute(1, 2, 0).contiguous(), -1) @ v[828:2876].double().transpose(0, 1).contiguous()
    close(one[4].reshape(hkv, -1, d), spot, v)
    for nsplit in (2, 3, 8, 9, 16, 17, 33, 64, 0):
        print("splits", h, hkv, d, nsplit, flush=True)
        close(_cabi.attn_paged_decode(q, k, v, table, rows, ind, nsplit=nsplit), one, v)


@pytest.mark.parametrize("h,hkv,seq", [(16, 4, 1), (16, 4, 2), (8, 8, 5), (6, 3, 3), (24, 8, 1)])
def test_dense_splits(h, hkv, seq):
    g = torch.Generator().manual_seed(seq)
    n, b = 300, 3
    q, k, v = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((b, h, seq, 128), (b, hkv, n, 128), (b, hkv, n, 128)))
    positions = torch.arange(n - seq, n, device="cuda")
    one = _cabi.attn_decode(q, k, v, positions, nsplit=1)
    for nsplit in (2, 5, 8, 64):
        close(_cabi.attn_decode(q, k, v, positions, nsplit=nsplit), one, v)
    codes, steps = _cabi.attn_decode(q, k, v, positions, nsplit=1, quantized=True)[:2]
    got = codes.double().reshape(b * seq, -1) * steps.double().reshape(-1, 1)
    # (an int8 step either side of the bf16 row that it was made from)
    assert bool(((got - one.double().reshape(b * seq, -1)).abs() <= 0.5001 * steps.double().reshape(-1, 1)).all())


def test_a_workspace_that_starts_off_the_vector_grid():
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((2, 16, 64), (600, 4, 64), (600, 4, 64)))
    table = torch.arange(600, dtype=torch.int32).reshape(2, 300).cuda()
    rows, ind = torch.arange(2, dtype=torch.int32).cuda(), torch.tensor([0, 300, 600], dtype=torch.int32).cuda()
    want = _cabi.attn_paged_decode(q, k, v, table, rows, ind, nsplit=7)
    room = torch.zeros(1 << 20, device="cuda")
    for off in (2, 6):
        got = _cabi.attn_paged_decode(q, k, v, table, rows, ind, nsplit=7, o_part_buf=room[off:])
        assert torch.equal(got, want)
