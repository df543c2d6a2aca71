"""A NaN in a query or key of the kernels for few rows and of the general ones: the rows that see it are NaN from end to
end, all others are bit for bit what they are without it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, NAN = "cuda", float("nan")


def _randn(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).to(DEV)


def _check(run, tensor, place, hit, what):
    """``run()`` gives ``[rows, heads, d]``; ``hit [rows, heads]`` of them see the NaN that goes to ``tensor[place]``."""
    clean = run()
    assert clean.isfinite().all(), what
    tensor[place] = NAN
    got, hit = run(), hit[..., None].expand_as(clean).to(clean.device)
    assert got[hit].isnan().all(), f"{what}: {int((~got[hit].isnan()).sum())} of {int(hit.sum())} values are not NaN"
    assert torch.equal(got[~hit], clean[~hit]), f"{what}: rows that do not see it changed"


def _heads(rows, h, row, heads):
    hit = torch.zeros(rows, h, dtype=torch.bool)
    hit[row, heads] = True
    return hit


@pytest.mark.parametrize("h,g,d", [(8, 2, 128), (8, 1, 128), (16, 1, 128), (8, 2, 64), (6, 2, 32), (4, 4, 256)])
@pytest.mark.parametrize("nsplit", [0, 1, 5])
@pytest.mark.parametrize("where", ["q", "k"])
@pytest.mark.parametrize("masked", [False, True])
def test_paged_decode(h, g, d, nsplit, where, masked):
    from astrai_amd.extension import _cabi
    lens = [40, 300, 1]
    q, k, v = _randn(3, h, d), _randn(sum(lens), g, d, seed=1), _randn(sum(lens), g, d, seed=2)
    ends = torch.tensor([0] + lens).cumsum(0).int()
    table = torch.zeros(3, 320, dtype=torch.int32)
    for i, m in enumerate(lens):
        table[i, :m] = ends[i] + torch.arange(m)
    args = [t.to(DEV) for t in (table, torch.arange(3, dtype=torch.int32), ends)]
    mask = torch.ones(3, 320, dtype=torch.bool, device=DEV) if masked else None
    run = lambda: _cabi.attn_paged_decode(q, k, v, *args, nsplit=nsplit, mask=mask).view(3, h, d)
    rep = h // g
    if where == "q":
        _check(run, q, (1, h - 1, 3), _heads(3, h, 1, slice(h - 1, h)), "query")
    else:
        _check(run, k, (40 + 20, 0, 5), _heads(3, h, 1, slice(0, rep)), "key")


@pytest.mark.parametrize("seq", [1, 2])
@pytest.mark.parametrize("nsplit", [1, 4])
@pytest.mark.parametrize("where", ["q", "k"])
def test_dense_decode(seq, nsplit, where):
    from astrai_amd.extension import _cabi
    b, h, g, d, length = 2, 8, 2, 128, 256
    q, k, v = _randn(b, h, seq, d), _randn(b, g, length, d, seed=1), _randn(b, g, length, d, seed=2)
    pos = torch.arange(seq, device=DEV) + 100
    run = lambda: _cabi.attn_decode(q, k, v, pos, nsplit=nsplit).view(b * seq, h, d)
    if where == "q":
        _check(run, q, (1, 6, 0, 9), _heads(b * seq, h, seq, slice(6, 7)), "query")
    else:
        _check(run, k, (1, 1, 99 + seq, 9), _heads(b * seq, h, b * seq - 1, slice(4, 8)), "key of the last token alone")


@pytest.mark.parametrize("h,g,d", [(6, 2, 32), (4, 4, 256), (8, 2, 64)])
@pytest.mark.parametrize("nsplit", [1, 3])
@pytest.mark.parametrize("where", ["q", "k"])
def test_paged_prompt_of_the_general_kernel(h, g, d, nsplit, where):
    from astrai_amd.extension import _cabi
    n, m = 70, 150
    q, k, v = _randn(n, h, d), _randn(m, g, d, seed=1), _randn(m, g, d, seed=2)
    args = [torch.arange(m, dtype=torch.int32, device=DEV)[None], torch.zeros(1, dtype=torch.int32, device=DEV),
            torch.tensor([0, m], dtype=torch.int32, device=DEV), *_cabi.paged_prefill_schedule([n], DEV)]
    mask = torch.ones(1, m, dtype=torch.bool, device=DEV) if d == 64 else None    # (a mask: the general kernel)
    run = lambda: _cabi.attn_paged_prefill(q, k, v, *args, mask=mask, causal_offset=0, nsplit=nsplit).view(n, h, d)
    if where == "q":
        _check(run, q, (33, 2, 3), _heads(n, h, 33, slice(2, 3)), "query")
    else:    # key 120: rows 40 and later see it
        _check(run, k, (120, g - 1, 3), _heads(n, h, slice(40, n), slice(h - h // g, h)), "key")


@pytest.mark.parametrize("softcap", [0.0, 20.0])
@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("nsplit", [1, 3])
@pytest.mark.parametrize("where", ["q", "k"])
def test_grouped_rows(softcap, sink, nsplit, where):
    from astrai_amd.extension import _mix
    s = _mix.GqaShape(8, 2, 64, 64, 64, 64 ** -0.5, softcap, sink)
    b, seq, length = 2, 3, 600
    proj, cache = _randn(b * seq, s.heads * s.dk), _randn(b, length, s.cache_cols, seed=1)
    pos = torch.arange(seq, device=DEV) + 500
    run = lambda: _mix.gqa_rows(proj, s, -1, cache, pos, True, nsplit).view(b * seq, s.heads, s.vp)
    if where == "q":
        _check(run, proj, (4, 7 * s.dk + 5), _heads(b * seq, s.heads, 4, slice(7, 8)), "query")
    else:    # a key of group 0 in sequence 1 that the last token alone sees
        _check(run, cache, (1, 502, 5), _heads(b * seq, s.heads, b * seq - 1, slice(0, 4)), "key")


@pytest.mark.parametrize("nsplit", [1, 3])
def test_latent_rows(nsplit):
    from astrai_amd.extension import _mix
    s = _mix.LatentShape(4, 64, 32, 128, 64, 128, 1 << 20, 96 ** -0.5)
    b, seq, length = 2, 3, 600
    proj, cache = _randn(b * seq, s.q_cols + 8), _randn(b, length, s.cache_cols, seed=1)
    w, q_abs = _randn(s.heads * (s.dn + s.vp), s.rp, seed=2), _randn(b * seq, s.heads, s.rp, seed=3)
    pos = torch.arange(seq, device=DEV) + 500
    run = lambda: _mix.latent_rows(proj, s, s.q_cols, w, cache, pos, q_abs.clone(), nsplit).view(b * seq, s.heads, s.vp)
    _check(run, q_abs, (4, 2, 7), _heads(b * seq, s.heads, 4, slice(2, 3)), "query")
