"""Products of few rows that leave planes for the norm behind them, inside whole models: every output projection without a bias
and every feed-forward, in prompts, steps, captured steps, passes of a loop and layers without a feed-forward."""

import pytest
import torch

import lugitar_helpers as LH
import sarulix_helpers as SH
from astrai_amd.extension import _mix
from astrai_amd.model import LugitarConfig, LugitarLM, SarulixLM, architecture_of, mixers
from oracle import lugitar_oracle as L
from oracle import sarulix_oracle as S

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = 6e-2   # bf16, the worst token's error over all layers, as in the models' own tests


def sarulix():
    wide = dict(heads=16, kv_heads=4, dim=24, vdim=128)
    cfg = SH.config([SH.delta(**wide, ff=2048), SH.rglru(width=2048, blocks=16), SH.attention(**wide, ff=2048), SH.delta(**wide),
                     SH.rglru(width=2048, blocks=16, ff=2304)], loop=(1, 4, 2))
    w = SH.tensors(cfg, 3)
    with torch.device(DEV):
        model = SarulixLM(architecture_of(cfg).configure(cfg, w)).to(torch.bfloat16).eval()
    return cfg, w, model.load_tensors(w), S.forward


def lugitar():
    cfg = LH.config([LH.latent(heads=16, vdim=128, window=None, ff=2048), LH.lightning(heads=16, vdim=128, decay=(0.5, 0.93, 0.9995, 0.97) * 4, ff=2048),
                     LH.latent(heads=16, dim=32, vdim=128, window=29, kv_from=0, ff=None),
                     LH.lightning(heads=16, dim=16, vdim=128, decay=(0.9,) * 16, ff=None)])
    w = LH.tensors(cfg, 3)
    with torch.device(DEV):
        model = LugitarLM(LugitarConfig.from_dict(cfg)).to(torch.bfloat16).eval()
    return cfg, w, model.load_tensors(w), L.forward


def logits(model, ids, cuts):
    cache, out, lo = model.new_cache(ids.size(0), ids.size(1)), [], 0
    for n in cuts:
        out.append(model(ids[:, lo:lo + n].to(DEV), cache)["logits"].float().cpu())
        cache.advance(n)
        lo += n
    return torch.cat(out, 1)


@pytest.mark.parametrize("family", [sarulix, lugitar])
def test_planes_and_whole_products_agree(family, monkeypatch):
    cfg, weights, model, oracle = family()
    ids = torch.randint(0, cfg["vocab"], (2, 40), generator=torch.Generator().manual_seed(1))
    want = torch.stack([oracle(cfg, weights, row) for row in ids])
    seen, parts = [], _mix.few_rows_parts
    monkeypatch.setattr(_mix, "few_rows_parts", lambda x, w, n: seen.append(w.data_ptr()) or parts(x, w, n))
    outputs = {layer.mix.o.weight.data_ptr() for layer in model.layers if layer.mix.o.bias is None}
    outputs |= {layer.mlp.down.weight.data_ptr() for layer in model.layers if layer.mlp is not None}
    assert len({type(layer.mix) for layer in model.layers if layer.mix.o.bias is None}) == 2   # (grouped attention's has one)
    for cuts in ([30, 1, 1, 8], [1] * 40, [32, 8]):   # (at most 64 rows)
        print(family.__name__, cuts[:3], flush=True)
        seen.clear()
        planes = logits(model, ids, cuts)
        assert set(seen) == outputs and len(seen) >= len(cuts) * len(outputs)
        with monkeypatch.context() as m:
            m.setattr(mixers, "parts_of", lambda *a: 1)
            count = len(seen)
            whole = logits(model, ids, cuts)
            assert len(seen) == count
        for got, to in ((planes, want), (whole, want), (planes, whole)):
            assert SH.relative_rms(got.flatten(0, 1), to.flatten(0, 1)) < TOL


@pytest.mark.parametrize("family", [sarulix, lugitar])
def test_captured_steps_repeat_the_eager_ones(family):
    cfg, _, model, _ = family()
    ids = torch.randint(0, cfg["vocab"], (2, 40), generator=torch.Generator().manual_seed(2)).to(DEV)
    cache, ref = model.new_cache(2, 40), model.new_cache(2, 40)
    for c in (cache, ref):
        model(ids[:, :20], c)
        c.advance(20)
    tok, pos = ids[:, 20:21].clone(), torch.full((1,), 20, device=DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        model(tok, model.new_cache(2, 40), pos)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = model(tok, cache, pos)["logits"]
    for i in range(20, 40):
        tok.copy_(ids[:, i:i + 1])
        pos.fill_(i)
        graph.replay()
        got = out.clone()
        cache.advance(1)
        want = model(ids[:, i:i + 1], ref)["logits"]
        ref.advance(1)
        assert torch.equal(got, want), i
