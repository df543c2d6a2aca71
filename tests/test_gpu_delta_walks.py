"""The chunked delta rule where its walk changes: up to 512 blocks of 16 value columns the waves of a workgroup share the
key channels, past that each takes all of them. The same sequences on both sides of the line, chunk counts of every
remainder of the walk's four turns, ragged last chunks. (Each side against the rule in 64 bits:
test_gpu_sarulix_ops.py.)"""
import pytest

from test_gpu_sarulix_ops import BF16, Delta, log, relative_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cuts", [[81], [64, 33, 5], [50, 1]], ids=str)
@pytest.mark.parametrize("shape", [(16, 8, 32, 32), (8, 4, 64, 64), (4, 2, 128, 128), (2, 2, 256, 256)], ids=str)
def test_both_walks(shape, cuts):
    heads, _, _, v = shape
    assert 16 * heads * v // 16 == 512
    log("delta walks", shape, cuts)
    runs = []
    for batch in (17, 16):
        c = Delta(shape, 3, BF16, sum(cuts), batch=17, seed=sum(cuts))
        for name in ("q", "k", "v", "b", "z", "gate", "state", "ring"):
            setattr(c, name, getattr(c, name)[:batch].contiguous())
        c.batch = batch
        runs.append((c.run(cuts, "chunk")[:16], c.state[:16].cpu()))
    (general, s_general), (split, s_split) = runs
    # Both multiply the same two-term images; the state as two bf16 terms misses 2^-17 of itself per product, three
    # products to a chunk, at most 8 chunks: 2 sides x 8 x 3 x 2^-17. Outputs are rounded to bf16 on top.
    assert relative_rms(s_split.reshape(16, -1), s_general.reshape(16, -1).double()) < 48 * 2.0 ** -17
    assert relative_rms(split.reshape(16, -1), general.reshape(16, -1).double()) < 2.0 ** -8


def test_an_infinite_value_stays_in_its_column():
    """One value is infinite: its column's state and every other column's outputs are what they are without the wave
    split as well: the column is lost from that chunk on, the others are finite."""
    c = Delta((2, 1, 64, 64), 1, BF16, 70, seed=3)
    c.v[0, 37, 0, 5] = float("inf")
    for w in c.cw:
        w[:] = 1.0
    got = c.run([70], "chunk").reshape(70, 2, 64)
    state = c.state.cpu()[0]
    assert got[:32].isfinite().all() and got[:, 1].isfinite().all() and state[1].isfinite().all()
    assert not state[0, :, 5].isfinite().any()
    state[0, :, 5] = 0.0
    assert state.isfinite().all()
