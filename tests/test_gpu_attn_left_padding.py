"""Prompt attention whose mask hides a row's first tiles of keys (padding in front), at several scales: the rows are softmax
attention over the keys they may attend, whatever the rounding of the scale times a hidden key's stand-in for -inf; a row
that may attend none is zero."""
import pytest
import torch

from test_gpu_attn_nonfinite import _check, _reference

pytestmark = pytest.mark.gpu
DEV = "cuda"
PADDING = (0, 31, 32, 64, 70, 130, 200)


@pytest.mark.parametrize("h,g,d", [(4, 2, 128), (8, 2, 128), (8, 1, 128), (4, 2, 64)])
@pytest.mark.parametrize("scale", [0.03, 0.05, 0.1, 0.125, 0.2, 0.6931472, 1.0])
@pytest.mark.parametrize("causal", [False, True])
def test_padding_in_front(h, g, d, scale, causal):
    from astrai_amd.extension import _cabi
    n = m = 200
    r = torch.Generator().manual_seed(d + h)
    b = len(PADDING)
    q, k, v = (torch.randn(*s, generator=r).to(torch.bfloat16) for s in ((b, n, h, d), (b, m, g, d), (b, m, g, d)))
    q = q * (0.3 / scale / d ** 0.5)    # scores of some ones, whatever the scale
    mask = torch.arange(m)[None, :] >= torch.tensor(PADDING)[:, None]
    got = _cabi.attn_prefill_qkv(*(t.to(DEV) for t in (q, k, v)), mask=mask.to(DEV), causal_offset=0 if causal else -1,
                                 scale=scale, layout=_cabi.BLHD)
    for i in range(b):
        seen = mask[i][None, :].expand(n, m)
        if causal:
            seen = seen & (torch.arange(m)[None, :] <= torch.arange(n)[:, None])
        want, weight = _reference(q[i].double() * (scale * d ** 0.5), k[i], v[i], seen)
        assert (got[i].cpu()[~seen.any(-1)] == 0).all(), f"{PADDING[i]} hidden: a row without a key is not zero"
        _check(got[i], want, weight, f"{PADDING[i]} hidden")
