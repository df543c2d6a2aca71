"""The start of an int8 forward in one launch (embedding rows, their norm and codes, rotary rows): the bits of its parts."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one workgroup per row below 512 rows and past 4096 values, one wave per row else
@pytest.mark.parametrize("shape,width,pairs,dtype", [((1, 1), 8, 1, torch.bfloat16), ((3, 5), 2048, 64, torch.float32),
                                                     ((32, 1), 2048, 64, torch.bfloat16), ((1, 511), 72, 32, torch.bfloat16),
                                                     ((2, 256), 1000, 3, torch.float32), ((5, 1003), 512, 64, torch.bfloat16),
                                                     ((4, 2100), 4096, 64, torch.bfloat16), ((1, 600), 8192, 48, torch.float32)])
def test_same_bits_as_its_parts(shape, width, pairs, dtype):
    from astrai_amd.extension import _cabi
    print(f"case {shape} {width}", flush=True)
    r = torch.Generator().manual_seed(width + shape[1])
    vocab = 300
    table, weight = (torch.randn(*s, generator=r).bfloat16().to(DEV) for s in ((vocab, width), (width,)))
    freqs = torch.randn(shape[1] + 70, pairs, 2, generator=r).to(dtype).to(DEV)
    ids = torch.randint(0, vocab, shape, generator=r).to(DEV)
    ids.view(-1)[0], ids.view(-1)[-1] = vocab - 1, 0
    positions = torch.arange(70, 70 + shape[1], device=DEV).flip(0).contiguous()
    x, xq, s, rotary = _cabi.embed_rmsnorm_quantize_int8(ids, table, weight, 1e-5, freqs, positions)
    want = F.embedding(ids, table)
    wq, ws = _cabi.add_rmsnorm_quantize_int8(want, weight, 1e-5)[:2]
    assert x.shape == want.shape and torch.equal(x, want)
    assert torch.equal(xq, wq) and torch.equal(s, ws)
    assert torch.equal(rotary, freqs.index_select(0, positions).unsqueeze(0).float())


@pytest.mark.parametrize("rows", [4, 700])
def test_outside_the_tables(rows):
    """Nothing is read there: rows of NaN, the others as ever."""
    from astrai_amd.extension import _cabi
    r = torch.Generator().manual_seed(rows)
    table, weight = (torch.randn(*s, generator=r).bfloat16().to(DEV) for s in ((50, 256), (256,)))
    freqs = torch.randn(20, 16, 2, generator=r).to(DEV)
    ids = torch.randint(0, 50, (1, rows), generator=r).to(DEV)
    ids[0, 1], ids[0, 2] = 50, -1
    positions = torch.tensor([0, 20, 19, -1, 1 << 40], device=DEV)
    x, _, _, rotary = _cabi.embed_rmsnorm_quantize_int8(ids, table, weight, 1e-5, freqs, positions)
    bad = torch.zeros(rows, dtype=torch.bool, device=DEV)
    bad[1:3] = True
    assert x[0, bad].isnan().all() and torch.equal(x[0, ~bad], F.embedding(ids[0, ~bad], table))
    assert rotary[0, [1, 3, 4]].isnan().all() and torch.equal(rotary[0, [0, 2]], freqs[[0, 19]])


def test_model_takes_it_and_leaves_observed_embeddings_alone():
    from astrai_amd.extension import w8a8
    from astrai_amd.model import AutoRegressiveLM, AutoRegressiveLMConfig, fuse_int8_weights
    torch.manual_seed(0)
    model = AutoRegressiveLM(AutoRegressiveLMConfig(hidden_size=512, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2,
                                                    intermediate_size=1024, vocab_size=128, max_position_embeddings=64)).to(DEV).bfloat16()
    fuse_int8_weights(model)
    ids = torch.randint(0, 128, (2, 9), device=DEV)
    with torch.no_grad(), w8a8.int8_autocast(True):
        assert model._start_fused_int8(ids, torch.arange(9, device=DEV)) is not None
        got = model(ids, model.new_cache(2, 16))["logits"]
        calls = []
        hook = model.embed_tokens.register_forward_hook(lambda m, a, o: calls.append(o.shape))
        seen = model(ids, model.new_cache(2, 16))["logits"]
        hook.remove()
        assert calls == [(2, 9, 512)] and torch.equal(seen, got)
        model.embed_tokens.forward = lambda t: F.embedding(t, model.embed_tokens.weight) * 0
        assert not torch.equal(model(ids, model.new_cache(2, 16))["logits"], got)
        del model.embed_tokens.forward
        assert torch.equal(model(ids.int(), model.new_cache(2, 16))["logits"], got)   # (another type of ids: the plain way)
    assert model._start_fused_int8(ids, torch.arange(9, device=DEV)) is None   # the policy is off


@pytest.mark.parametrize("rows,width", [(4, 256), (4, 8192), (700, 256), (700, 4096)])
def test_a_row_of_nan_has_such_a_step_where_the_norm_goes_out(rows, width):
    from astrai_amd.extension import _cabi
    r = torch.Generator().manual_seed(rows)
    x, weight = (torch.randn(*s, generator=r).bfloat16().to(DEV) for s in ((rows, width), (width,)))
    wq, ws, _, wy = _cabi.add_rmsnorm_quantize_int8(x, weight, 1e-5, None, True)
    x[1, 5] = float("nan")
    good = torch.arange(rows, device=DEV) != 1
    xq, s, _, y = _cabi.add_rmsnorm_quantize_int8(x, weight, 1e-5, None, True)
    assert s[1].isnan().all() and y[1].isnan().all()
    assert torch.equal(s[good], ws[good]) and torch.equal(xq[good], wq[good]) and torch.equal(y[good], wy[good])
    s = _cabi.add_rmsnorm_quantize_int8(x, weight, 1e-5)[1]
    assert torch.isfinite(s).all() and torch.equal(s[good], ws[good])


@pytest.mark.parametrize("batch,seq,cached", [(2, 9, True), (2, 9, False), (1, 600, True), (5, 1, True)])
def test_logits_of_what_is_outside_the_tables(batch, seq, cached):
    """NaN for such a token and for one at such a place; what does not attend to it as ever."""
    from astrai_amd.extension import w8a8
    from astrai_amd.model import AutoRegressiveLM, AutoRegressiveLMConfig, fuse_int8_weights
    torch.manual_seed(0)
    places = 640
    model = AutoRegressiveLM(AutoRegressiveLMConfig(hidden_size=512, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2,
                                                    intermediate_size=1024, vocab_size=128, max_position_embeddings=places)).to(DEV).bfloat16()
    fuse_int8_weights(model)
    ids = torch.randint(0, 128, (batch, seq), device=DEV)
    run = lambda t, at=None: model(t, model.new_cache(batch, 1300) if cached else None, at)["logits"]  # noqa: E731
    with torch.no_grad(), w8a8.int8_autocast(True):
        want = run(ids)
        assert torch.isfinite(want).all()
        for bad in (128, -1, 1 << 40):
            wrong = ids.clone()
            wrong[batch - 1, seq // 2] = bad
            assert model._start_fused_int8(wrong, torch.arange(seq, device=DEV)) is not None
            got = run(wrong)
            assert got[batch - 1, seq // 2].isnan().all()
            assert torch.equal(got[:batch - 1], want[:batch - 1]) and torch.equal(got[batch - 1, :seq // 2], want[batch - 1, :seq // 2])
        at = torch.arange(places - seq // 2, places - seq // 2 + seq, device=DEV)
        got = run(ids, at)
        assert torch.isfinite(got[:, :seq // 2]).all() and got[:, seq // 2:].isnan().all()
