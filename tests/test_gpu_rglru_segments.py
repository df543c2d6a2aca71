"""The gated linear recurrence over the segments that the default rule cuts a sequence into: more segments than the eight
whose decays are fetched at once, last segments that are ragged, short or empty, on either side of the line past which
nothing is cut. Against the same kernel walking each sequence whole."""
import pytest
import torch

from astrai_amd.extension import _mix
from lugitar_helpers import relative_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks,bp", [(2, 64), (3, 160), (2, 256), (1, 1024)])
@pytest.mark.parametrize("batch,seq", [(1, 1), (1, 65), (1, 700), (2, 1089), (5, 1000), (1, 2500), (59, 130)])
def test_default_segments(blocks, bp, batch, seq):
    nseg, cols = _mix.rglru_nseg(batch, blocks, bp, seq), blocks * bp
    assert 1 <= nseg <= -(-seq // 64)
    print("segments", blocks, bp, batch, seq, nseg, flush=True)
    g = torch.Generator().manual_seed(seq)

    def rand(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).cuda()

    u, proj = rand(batch * seq, cols).bfloat16(), rand(batch * seq, 2 * cols).bfloat16()
    w = [rand(blocks, bp, bp, std=bp ** -0.5).bfloat16() for _ in range(2)]
    gates, start = [rand(cols), rand(cols), -rand(cols).abs() - 0.01], rand(batch, cols)
    runs = []
    for n in (None, 1):
        state = start.clone()
        runs.append((_mix.rglru(u, proj, 0, *w, *gates, state, matrix=True, nseg=n), state))
    # Decays at most 1, fp32: the sums only associate differently, 2^-24 for each of the segments' two roundings and
    # as much again per tile; outputs are rounded to bf16 on top.
    bound = 4 * -(-seq // 64) * 2.0 ** -24
    assert relative_rms(runs[0][1].cpu(), runs[1][1].cpu().double()) <= bound
    assert relative_rms(runs[0][0].cpu(), runs[1][0].cpu().double()) <= 2.0 ** -9 + bound
