"""Ragged prompts over a pool whose schedule has few tiles: the keys of a block of queries in several parts, each a
workgroup's, merged by a second launch. Against 64-bit attention, and the same call with one part."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

HEADS = [(16, 16, 64), (4, 2, 64), (16, 4, 64), (32, 4, 64), (16, 16, 128)]
# (query rows, keys) of each sequence, width of the table; the parts end at multiples of 64 keys
SHAPES = {
    "long": ([(130, 1000), (64, 1088), (1, 1025)], 1088),
    "mixed": ([(33, 33), (40, 900), (64, 64), (1, 1), (60, 64 * 9 + 1)], 1500),
    "wide table": ([(100, 130), (64, 200), (65, 65)], 4096),
    "no keys": ([(70, 0), (90, 20), (128, 700)], 703),
    "one block each": ([(65, 65 + 64 * k) for k in (3, 9)], 1024),
}


def _case(h, g, d, seqs, width, seed, scale=1.0):
    r = torch.Generator().manual_seed(seed)
    n, m = sum(a for a, _ in seqs), sum(b for _, b in seqs)
    q = (torch.randn(n, h, d, generator=r) * scale).bfloat16()
    k, v = (torch.randn(m + 5, g, d, generator=r).bfloat16() for _ in range(2))
    order = torch.randperm(m + 5, generator=r)[:m].int()
    table, at = torch.full((len(seqs) + 1, width), -1, dtype=torch.int32), 0
    for i, (_, b) in enumerate(seqs):
        table[i + 1, :b] = order[at:at + b]
        at += b
    rows = torch.arange(1, len(seqs) + 1, dtype=torch.int32)
    kv = torch.tensor([0] + [b for _, b in seqs]).cumsum(0).int()
    return q, k, v, table, rows, kv


def _exact(q, k, v, table, seqs, causal):
    out, at = torch.zeros(q.shape, dtype=torch.float64), 0
    for i, (n, m) in enumerate(seqs):
        if m:
            at_k = table[i + 1, :m].long()
            rep = q.size(1) // k.size(1)
            kk, vv = (t[at_k].double().repeat_interleave(rep, 1) for t in (k, v))
            s = torch.einsum("nhd,mhd->hnm", q[at:at + n].double(), kk) * q.size(2) ** -0.5
            if causal:
                s = s.masked_fill(torch.arange(m)[None] > torch.arange(n)[:, None] + m - n, float("-inf"))
            p = torch.softmax(s, -1).nan_to_num(0.0)
            out[at:at + n] = torch.einsum("hnm,mhd->nhd", p, vv)
        at += n
    return out


def _call(case, seqs, causal, nsplit=0):
    from astrai_amd.extension import _cabi
    dev = [t.to(DEV) for t in case]
    sched = _cabi.paged_prefill_schedule([n for n, _ in seqs], DEV)
    return lambda: _cabi.attn_paged_prefill(*dev, *sched, causal_offset=0 if causal else -1, nsplit=nsplit)


def _close(got, want, what):
    # the result's rounding (2^-9 of it), and probabilities of two bf16 terms, 2^-16 of values up to 6
    err = (got.double().cpu() - want).abs()
    assert (err <= 2.0 ** -8 * want.abs() + 6 * 2.0 ** -14).all(), (what, err.max())


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("h,g,d", HEADS)
def test_parts_agree_with_64_bits(h, g, d, shape, causal):
    seqs, width = SHAPES[shape]
    case = _case(h, g, d, seqs, width, seed=h + d)
    want = _exact(*case[:4], seqs, causal)
    for nsplit in (0, 2, 3, 16):
        _close(_call(case, seqs, causal, nsplit)(), want, nsplit)


@pytest.mark.parametrize("h,g,d", HEADS)
def test_error_is_no_larger_than_without_parts(h, g, d):
    seqs, width = SHAPES["long"]
    case = _case(h, g, d, seqs, width, seed=9, scale=4.0)   # (peaked rows: maxima that differ from part to part)
    want = _exact(*case[:4], seqs, True)
    whole, parts = ((_call(case, seqs, True, n)().double().cpu() - want) for n in (1, 16))
    # both are the rounding of the result but for what fp32 and P's second term leave
    assert parts.norm() <= whole.norm() * 1.01
    assert parts.abs().max() <= whole.abs().max() * 1.01 + 2.0 ** -14


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("h,g,d", [(16, 16, 64), (16, 16, 128)])
def test_what_is_not_a_number_reaches_the_same_rows(h, g, d, bad):
    seqs, width = SHAPES["long"]
    case = _case(h, g, d, seqs, width, seed=3)
    case[1][case[3][1, 950].long()] = bad     # a key of the first sequence's last part, that its last rows see
    whole, parts = (_call(case, seqs, True, n)() for n in (1, 16))
    assert torch.equal(torch.isnan(whole), torch.isnan(parts)) and torch.isnan(parts).any() and torch.isfinite(parts).any()


def test_missing_slots_and_a_row_that_is_no_request():
    seqs, width = SHAPES["long"]
    q, k, v, table, rows, kv = _case(16, 16, 64, seqs, width, seed=4)
    table[2, 100] = table[2, 700] = -1                     # attended as zeros
    rows = rows.clone()
    rows[2] = 99                                           # no keys
    case = (q, k, v, table, rows, kv)
    whole, parts = (_call(case, seqs, True, n)() for n in (1, 16))
    assert (parts[-1] == 0).all()
    assert ((parts.float() - whole.float()).abs() <= 2.0 ** -7 * whole.float().abs() + 6 * 2.0 ** -13).all()


def test_captured_and_with_a_workspace_on_any_float():
    from astrai_amd.extension import _cabi
    seqs, width = SHAPES["long"]
    case = _case(16, 16, 64, seqs, width, seed=5)
    call = _call(case, seqs, True)
    want = call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = call()
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(call(), want)
    lib = _cabi.load()
    q, k, v, table, rows, kv = (t.to(DEV) for t in case)
    qo, tb, ti = _cabi.paged_prefill_schedule([n for n, _ in seqs], DEV)
    need = lib.astrai_w8a8_attn_paged_rows_workspace_floats(tb.numel(), 16, 16, 64, 16, 1)
    ws = torch.full((need + 2,), float("nan"), device=DEV)
    out = torch.empty_like(q)
    _cabi._check(lib.astrai_w8a8_attn_paged_rows_bf16(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr(), rows.data_ptr(), kv.data_ptr(), qo.data_ptr(), tb.data_ptr(),
        ti.data_ptr(), None, 0, 0, 0, 0, 0, ws.data_ptr() + 4, need, out.data_ptr(), tb.numel(), 16, 16, 64, k.size(0),
        table.size(0), table.size(1), 1, 16, 64 ** -0.5, _cabi._stream(q)), lib)
    assert torch.isnan(ws[0]) and torch.isnan(ws[-1])
    _close(out, _exact(*case[:4], seqs, True), "any float")
