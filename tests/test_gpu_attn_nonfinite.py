"""NaN and infinities in the queries and keys of prompt attention: a row whose scores hold a NaN, or an infinity that wins,
is NaN as softmax in float64 has it; rows that do not see the place are what they are without it, rows that see no key zero."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, NAN, INF = "cuda", float("nan"), float("inf")
SHAPES = [(4, 4, 64), (4, 2, 64), (8, 2, 64), (8, 1, 64), (3, 3, 128), (4, 2, 128), (8, 2, 128), (8, 1, 128)]


def _reference(q, k, v, seen):
    """``q [n, h, d]``, ``k``, ``v [m, g, d]``, ``seen [n, m]``; a row that sees nothing: zeros. Also sum p |v|."""
    rep = q.size(1) // k.size(1)
    q, k, v = (t.double().transpose(0, 1) for t in (q, k, v))
    k, v = k.repeat_interleave(rep, 0), v.repeat_interleave(rep, 0)
    s = ((q @ k.transpose(1, 2)) * q.size(-1) ** -0.5).masked_fill(~seen, -INF)
    p = torch.where(seen.any(-1)[:, None], torch.softmax(s, -1), 0.0)
    return (p @ v).transpose(0, 1), (p @ v.abs()).transpose(0, 1)


def _check(got, want, weight, what):
    # probabilities and output are rounded to bf16 once each (2^-8 at most); scores, exponentials and sums in fp32
    # are good for 2^-16 of sum p |v|: a tenth of the bound covers them
    got = got.double().cpu()
    assert torch.equal(got.isnan(), want.isnan()), f"{what}: NaN in {int(got.isnan().sum())} places of {int(want.isnan().sum())}"
    assert got.isinf().sum() == 0, what
    err, bound = (got - want).abs().nan_to_num(), (1.1 * 2.0 ** -8 * (weight + want.abs())).nan_to_num() + 1e-7
    assert (err <= bound).all(), f"{what}: worst {(err / bound).max().item():.2f} of the bound"


def _poisoned(n, m, h, g, d, where, value):
    r = torch.Generator().manual_seed(n + d)
    q, k, v = (torch.randn(*s, generator=r).to(torch.bfloat16) for s in ((n, h, d), (m, g, d), (m, g, d)))
    k[:3, :, 0] = 1.0    # an infinite query meets both signs
    k[3, :, 0] = -1.0
    if where == "q":
        q[n - 7, :, 0] = value
    else:
        k[m // 2, :, 0] = value
    return q, k, v


CASES = [(where, value) for where in ("q", "k") for value in (NAN, INF, -INF)]


@pytest.mark.parametrize("h,g,d", SHAPES)
@pytest.mark.parametrize("where,value", CASES)
def test_dense(h, g, d, where, value):
    from astrai_amd.extension import _cabi
    n, m = 150, 200
    q, k, v = _poisoned(n, m, h, g, d, where, value)
    newest = torch.arange(n) + m - n
    want, weight = _reference(q, k, v, torch.arange(m)[None, :] <= newest[:, None])
    got = _cabi.attn_prefill_qkv(*(t[None].to(DEV) for t in (q, k, v)), causal_offset=m - n, layout=_cabi.BLHD)
    _check(got[0], want, weight, "tensors")
    caches = [t.transpose(0, 1)[None].contiguous().to(DEV) for t in (q, k, v)]
    got = _cabi.attn_cache_rows(*caches, newest.to(DEV)).view(n, h, d)
    _check(got, want, weight, "cache")
    if _cabi.attn_prefill_supported(h, g, d):
        _check(_cabi.attn_prefill(*caches, newest.to(DEV)).view(n, h, d), want, weight, "cache, block kernel")


@pytest.mark.parametrize("h,g,d", SHAPES)
@pytest.mark.parametrize("where,value", CASES)
def test_paged(h, g, d, where, value):
    from astrai_amd.extension import _cabi
    n, m = 150, 200
    q, k, v = _poisoned(n, m, h, g, d, where, value)
    table = torch.arange(m, dtype=torch.int32)[None].to(DEV)
    args = [q.to(DEV), k.to(DEV), v.to(DEV), table, torch.zeros(1, dtype=torch.int32, device=DEV),
            torch.tensor([0, m], dtype=torch.int32, device=DEV), *_cabi.paged_prefill_schedule([n], DEV)]
    causal = torch.arange(m)[None, :] <= (torch.arange(n) + m - n)[:, None]
    _check(_cabi.attn_paged_prefill(*args, causal_offset=0, nsplit=1), *_reference(q, k, v, causal), "causal")
    if not _cabi.attn_prefill_supported(h, g, d):
        return    # (a mask keeps these shapes on the general kernel)
    mask = torch.rand(n, m, generator=torch.Generator().manual_seed(1)) < 0.5
    mask[:, m // 2] = torch.arange(n) % 3 != 0    # a third of the rows do not see the key
    mask[n - 9:n - 5] = False                     # rows that see nothing, the poisoned query's one of them
    mask[20:24] = False                           # rows that see that key alone
    mask[20:24, m // 2] = True
    got = _cabi.attn_paged_prefill(*args, mask=mask[None, None].to(DEV), causal_offset=-1)
    want, weight = _reference(q, k, v, mask)
    if value == -INF or value == INF:
        # a single visible score of -inf has no softmax; the kernels give zeros for it
        lone = want[20:24].isnan()
        want[20:24], weight[20:24] = torch.where(lone & (got[20:24].cpu() == 0), 0.0, want[20:24]), weight[20:24].nan_to_num()
    _check(got, want, weight, "mask")
