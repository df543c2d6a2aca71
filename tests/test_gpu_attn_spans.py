"""Prompt attention where byte offsets pass 2 and 4 GiB: a row that is missing (no slot, or past the newest key) reads as
zeros, never as another place of the pool or tensor."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("nbytes", [(1 << 31) + (1 << 20), (1 << 32) - 256, (1 << 32) - 128], ids=str)
@pytest.mark.parametrize("h,g,d", [(8, 2, 64), (2, 1, 64), (2, 2, 128), (8, 2, 128)])
def test_missing_slots_of_a_large_pool(h, g, d, nbytes):
    from astrai_amd.extension import _cabi
    slots = nbytes // (2 * g * d)
    print("large pool", h, g, d, slots, flush=True)
    r = torch.Generator().manual_seed(d)
    n = m = 150
    q, rows = torch.randn(n, h, d, generator=r).bfloat16().to(DEV), torch.randn(m, g, d, generator=r).bfloat16().to(DEV)
    sched = _cabi.paged_prefill_schedule([n], DEV)
    ints = [torch.zeros(1, dtype=torch.int32, device=DEV), torch.tensor([0, m], dtype=torch.int32, device=DEV), *sched]
    table = torch.arange(m, dtype=torch.int32, device=DEV)[None].clone()
    table[0, 40], table[0, 70] = -1, 2 ** 31 - 1
    want = _cabi.attn_paged_prefill(q, rows, rows, table, *ints, causal_offset=0, nsplit=1)
    # the same rows from both ends of the pool; everything else in it is NaN
    pool = torch.full((slots, g, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    pool[:75], pool[-75:] = rows[:75], rows[75:]
    table[0, 75:] += slots - m
    got = _cabi.attn_paged_prefill(q, pool, pool, table, *ints, causal_offset=0, nsplit=1)
    # (the same kernel but for the largest pool, whose shapes with P in two terms differ by an ulp: 2^-7)
    err = (got.float() - want.float()).abs()
    assert torch.isfinite(got).all() and (err <= 2.0 ** -7 * want.float().abs() + 2 * 5 * 2.0 ** -16).all()


def test_rows_past_the_newest_key_of_a_far_strided_tensor():
    from astrai_amd.extension import _cabi
    base = torch.full((1 << 31,), float("nan"), dtype=torch.bfloat16, device=DEV)
    q = torch.randn(1, 8, 40, 64, device=DEV).bfloat16()
    # whole blocks of 64 keys are fetched: of the rows behind the last, the second lies past 2^32 bytes
    for m in (65, 33, 2):
        stride = ((1 << 31) - 128) // m // 8 * 8
        k = torch.as_strided(base, (1, 2, m, 64), (8, 64, stride, 1))
        k.copy_(torch.randn(1, 2, m, 64, device=DEV))
        want = _cabi.attn_prefill_strided(q, k.contiguous(), k.contiguous(), _cabi.BHLD)
        got = _cabi.attn_prefill_strided(q, k, k, _cabi.BHLD)
        assert torch.isfinite(got).all() and torch.equal(got, want), m
        k.fill_(float("nan"))
