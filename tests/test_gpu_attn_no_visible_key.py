"""Causal paged prompts with far more query rows than keys: whole blocks of rows lie before the first key. They are zero,
the others softmax attention, for every number of token groups that a workgroup holds."""
import pytest
import torch

from test_gpu_attn_nonfinite import SHAPES, _check, _reference

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("h,g,d", SHAPES + [(4, 2, 32), (4, 2, 256)])
@pytest.mark.parametrize("lens", [[(200, 400)], [(1, 130), (64, 64), (0, 200), (33, 300)], [(65, 192)]], ids=str)
@pytest.mark.parametrize("masked", [False, True])
def test_more_rows_than_keys(h, g, d, lens, masked):
    from astrai_amd.extension import _cabi
    print("no visible key", h, g, d, lens, masked, flush=True)
    r = torch.Generator().manual_seed(d)
    kv, new = [a for a, _ in lens], [b for _, b in lens]
    slots, most = sum(kv) + 8, 256
    k, v = (torch.randn(slots, g, d, generator=r).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(sum(new), h, d, generator=r).to(torch.bfloat16)
    perm, at = torch.randperm(slots, generator=r), 0
    table = torch.full((len(kv), most), -1, dtype=torch.int32)
    want, weight = [], []
    for i, (m, n) in enumerate(lens):
        mine = perm[at:at + m]
        table[i, :m] = mine.int()
        at += m
        seen = torch.arange(max(m, 1))[None, :] <= (torch.arange(n) + m - n)[:, None]
        rows = q[sum(new[:i]):sum(new[:i + 1])]
        y, w = _reference(rows, k[mine], v[mine], seen) if m else (torch.zeros(n, h, d).double(),) * 2
        want.append(y)
        weight.append(w)
    args = [t.to(DEV) for t in (q, k, v, table, torch.arange(len(kv), dtype=torch.int32),
                                torch.tensor([0] + kv).cumsum(0).int())]
    mask = torch.ones(len(kv), most, dtype=torch.bool, device=DEV) if masked else None
    got = _cabi.attn_paged_prefill(*args, *_cabi.paged_prefill_schedule(new, DEV), mask=mask, causal_offset=0, nsplit=1)
    want, weight = torch.cat(want), torch.cat(weight)
    assert (got.cpu()[(weight == 0).all(-1)] == 0).all(), "a row without a key is not zero"
    _check(got, want, weight, "rows")
