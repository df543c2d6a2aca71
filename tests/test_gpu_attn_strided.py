"""The prompt attention kernel on tensors of any memory order and at the head shapes it shares with the
general kernel (head_dim 64; one query head per KV head), against softmax attention in float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

SHAPES = [(4, 4, 64), (6, 3, 64), (8, 2, 64), (8, 1, 64), (3, 3, 128), (4, 2, 128), (8, 2, 128), (8, 1, 128)]


def _reference(q, k, v, newest):
    """``q [b, n, h, d]``, ``k``, ``v [b, m, g, d]``; query i sees keys 0 .. newest[i]."""
    rep = q.size(2) // k.size(2)
    q, k, v = (t.double().cpu().transpose(1, 2) for t in (q, k, v))
    k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    s = (q @ k.transpose(-1, -2)) * q.size(-1) ** -0.5
    seen = torch.arange(k.size(2))[None, :] <= newest[:, None]
    p = torch.softmax(s.masked_fill(~seen, float("-inf")), -1).nan_to_num()
    return (p @ v).transpose(1, 2), (p @ v.abs()).transpose(1, 2)


def _check(got, want, weight, what):
    """Probabilities and output are rounded to bf16 once each (8 significant bits: a relative 2^-8 at most, half
    an ulp just above a power of two): 2^-8 of sum p |v| and of |y|. Scores, exponentials and sums in fp32 are
    good for 2^-16 of that sum: a tenth of the bound covers them many times over."""
    err = (got.double().cpu() - want).abs()
    assert torch.isfinite(got).all(), what
    bound = 1.1 * 2.0 ** -8 * (weight + want.abs())
    assert (err <= bound + 1e-7).all(), f"{what}: worst {(err / (bound + 1e-7)).max().item():.2f} of the bound"


def _tensors(b, n, m, h, g, d, seed):
    r = torch.Generator(device=DEV).manual_seed(seed)
    mk = lambda *size: torch.randn(*size, generator=r, device=DEV).to(torch.bfloat16)
    return mk(b, n, h, d), mk(b, m, g, d), mk(b, m, g, d)


@pytest.mark.parametrize("h,g,d", SHAPES)
@pytest.mark.parametrize("n,m", [(1, 1), (31, 31), (33, 64), (64, 65), (65, 65), (97, 128), (130, 130), (200, 333)])
def test_every_shape_and_edge(h, g, d, n, m):
    from astrai_amd.extension import _cabi
    q, k, v = _tensors(2, n, m, h, g, d, seed=n + m)
    for off in (m - n, -1, 0, m + 3):
        newest = torch.full((n,), m - 1) if off < 0 else (torch.arange(n) + off).clamp_max(m - 1)
        got = _cabi.attn_prefill_strided(q, k, v, _cabi.BLHD, off)
        _check(got, *_reference(q, k, v, newest), f"{h}/{g}x{d} {n} of {m} offset {off}")
    # arbitrary positions, one of them past the keys
    pos = torch.randint(0, m, (n,), generator=torch.Generator().manual_seed(5))
    pos[-1] = m + 7
    got = _cabi.attn_prefill_strided(q, k, v, _cabi.BLHD, positions=pos.to(DEV))
    _check(got, *_reference(q, k, v, pos.clamp_max(m - 1)), f"{h}/{g}x{d} {n} of {m} positions")


@pytest.mark.parametrize("h,g,d", [(2, 2, 64), (4, 2, 64), (4, 1, 64), (2, 2, 128), (4, 2, 128), (4, 1, 128), (8, 1, 128)])
@pytest.mark.parametrize("cached", [0, 31, 129])
def test_odd_and_even_tiles_blocks_and_rounds_of_the_rings(h, g, d, cached):
    """Every remainder of the walk: the last block of one tile or two, an odd block behind the pairs, none and several."""
    from astrai_amd.extension import _cabi
    for n in (32, 64, 96, 129, 161, 192, 224, 257, 289, 352, 417):
        q, k, v = _tensors(1, n, n + cached, h, g, d, seed=n)
        newest = torch.arange(n) + cached
        got = _cabi.attn_prefill_strided(q, k, v, _cabi.BLHD, cached)
        _check(got, *_reference(q, k, v, newest), f"{h}/{g}x{d} {n} behind {cached}")


@pytest.mark.parametrize("h,g,d", SHAPES)
def test_memory_orders_give_the_same_bits(h, g, d):
    from astrai_amd.extension import _cabi
    b, n = 2, 150
    q, k, v = _tensors(b, n, n, h, g, d, seed=h + d)
    want = _cabi.attn_prefill_strided(q, k, v, _cabi.BLHD, 0)
    heads_first = [t.transpose(1, 2).contiguous() for t in (q, k, v)]
    assert torch.equal(_cabi.attn_prefill_strided(*heads_first, _cabi.BHLD, 0), want)
    # views of one fused projection, read in place; with an odd row stride, copied
    for pad in (0, 8, 3):
        fused = torch.zeros(b, n, (h + 2 * g) * d + pad, device=DEV, dtype=torch.bfloat16)
        parts, at = [], 0
        for t in (q, k, v):
            cols = t.size(2) * d
            fused[..., at:at + cols] = t.reshape(b, n, cols)
            parts.append(fused[..., at:at + cols].unflatten(-1, (-1, d)))
            at += cols
        assert torch.equal(_cabi.attn_prefill_strided(*parts, _cabi.BLHD, 0), want), pad
    # through the entry with the reference's arguments, both layouts
    assert torch.equal(_cabi.attn_prefill_qkv(q, k, v, causal_offset=0, layout=_cabi.BLHD), want)
    assert torch.equal(_cabi.attn_prefill_qkv(*heads_first, causal_offset=0, layout=_cabi.BHLD).transpose(1, 2), want)
    # keys and values shared by the batch (stride 0)
    one = [t[:1].expand(b, -1, -1, -1) for t in (k, v)]
    assert torch.equal(_cabi.attn_prefill_strided(q, *one, _cabi.BLHD, 0)[0], want[0])


@pytest.mark.parametrize("h,g,d", [(4, 4, 64), (8, 4, 64), (8, 2, 64), (16, 2, 64), (4, 4, 128)])
def test_paged_block_kernel_equals_the_general_kernel(h, g, d):
    """Ragged sequences, empty ones, padding slots, a poisoned pool; an all-True mask keeps a call on the
    general kernel. Both carry P in 16 bits of mantissa (2^-16 of sum p |v|, |v| < 5) and round the output
    once: they differ by an ulp (2^-7 of |y| at most) where that falls across a rounding point."""
    from astrai_amd.extension import _cabi
    q_lens, kv_lens = [1, 64, 0, 33, 130, 7], [1, 64, 0, 95, 200, 3]
    r = torch.Generator().manual_seed(h * d)
    pool, b = sum(kv_lens) + 40, len(kv_lens)
    perm = torch.randperm(pool, generator=r)
    table, at = torch.full((b, 256), -1, dtype=torch.int32), 0
    for i, n in enumerate(kv_lens):
        table[i, :n] = perm[at:at + n].int()
        at += n
    table[4, 5] = -1
    table[4, 9] = pool + 4
    k, v = (torch.randn(pool, g, d, generator=r).to(torch.bfloat16) for _ in range(2))
    k[perm[at:]] = v[perm[at:]] = float("nan")
    q = torch.randn(sum(q_lens), h, d, generator=r).to(torch.bfloat16)
    args = [t.to(DEV) for t in (q, k, v, table, torch.arange(b, dtype=torch.int32),
                                torch.tensor([0] + kv_lens).cumsum(0).int())]
    sched = _cabi.paged_prefill_schedule(q_lens, DEV)
    for causal in (0, -1):
        got = _cabi.attn_paged_prefill(*args, *sched, causal_offset=causal, nsplit=1)
        want = _cabi.attn_paged_prefill(*args, *sched, causal_offset=causal, nsplit=1,
                                        mask=torch.ones(b, 256, dtype=torch.bool, device=DEV))
        assert torch.isfinite(got).all()
        err = (got.float() - want.float()).abs()
        assert (err <= 2.0 ** -7 * want.float().abs() + 2 * 5 * 2.0 ** -16).all(), err.max()


def test_nan_in_a_later_value_stays_within_its_block():
    """A value row that no query of a 32-token block sees does not reach the block's outputs."""
    from astrai_amd.extension import _cabi
    for h, g, d in SHAPES:
        q, k, v = _tensors(1, 256, 256, h, g, d, seed=1)
        v[0, 160] = float("nan")
        out = _cabi.attn_prefill_strided(q, k, v, _cabi.BLHD, 0)
        assert torch.isfinite(out[0, :160]).all() and out[0, 160:].isnan().all(), (h, g, d)


@pytest.mark.parametrize("h,g,d", SHAPES[:2] + SHAPES[4:6])
def test_tensors_off_the_16_byte_grid_that_count_as_contiguous(h, g, d):
    from astrai_amd.extension import _cabi
    q, k, v = _tensors(1, 70, 70, h, g, d, seed=d)
    want = _cabi.attn_prefill_strided(q, k, v, _cabi.BLHD, 0)
    shifted = [torch.cat((t.new_zeros(1), t.flatten()))[1:].view_as(t) for t in (q, k, v)]
    assert all(t.is_contiguous() and t.data_ptr() % 16 for t in shifted)
    assert torch.equal(_cabi.attn_prefill_strided(*shifted, _cabi.BLHD, 0), want)
    odd = [torch.as_strided(t, t.shape, (t.stride(0) + 1, *t.stride()[1:])) for t in (q, k, v)]   # of a batch of one
    assert all(t.is_contiguous() for t in odd)
    assert torch.equal(_cabi.attn_prefill_strided(*odd, _cabi.BLHD, 0), want)
    assert torch.equal(_cabi.attn_prefill_qkv(*shifted, causal_offset=0, layout=_cabi.BLHD), want)


def test_more_than_a_million_short_sequences():
    from astrai_amd.extension import _cabi
    b = (1 << 20) + 3
    q, k, v = (torch.randn(b, 2, n, 64, device=DEV).bfloat16() for n in (2, 1, 1))
    got = _cabi.attn_prefill_qkv(q, k, v, causal_offset=0, layout=_cabi.BLHD)
    for at in (0, 1 << 19, b - 5):
        part = slice(at, at + 5)
        assert torch.equal(got[part], _cabi.attn_prefill_qkv(q[part], k[part], v[part], causal_offset=0, layout=_cabi.BLHD))
