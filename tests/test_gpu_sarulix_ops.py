"""The kernels of grouped attention with a sink, the gated linear recurrence, the channel-wise delta rule and
their row operations, against the plain implementation in float64 on the same inputs."""

import pytest
import torch

from astrai_amd.extension import _mix
from astrai_amd.extension._mix import DeltaShape, GqaShape, pad_to
from astrai_amd.model.mixers import Rotation
from lugitar_helpers import relative_rms
from oracle import sarulix_oracle as S

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.float32: 1e-5, torch.bfloat16: 1e-2}
DTYPES = [torch.float32, torch.bfloat16]
BF16 = torch.bfloat16


def randn(g, *size, dtype=torch.float32, std=1.0):
    return (torch.randn(*size, generator=g) * std).to(dtype)


def gen(seed=0):
    return torch.Generator().manual_seed(seed)


def log(*what):
    print(*what, flush=True)


def padded(t, *sizes):
    """Zeros appended to the last axes."""
    out = t.new_zeros(*t.shape[:t.dim() - len(sizes)], *sizes)
    out[tuple(slice(0, n) for n in t.shape)] = t
    return out


# ---------------------------------------------------------------- row operations


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [1, 72, 101, 1024, 1028, 3000, 8192, 9000])
def test_sum_norm(width, dtype):
    g = gen(width)
    n, eps = 7, 1e-3
    w, vec = randn(g, width) + 1, randn(g, width)
    x, table, tokens = randn(g, n, width, std=3.0), randn(g, 11, width, dtype=dtype), torch.tensor([3, 0, 10, 3, 5, 5, 9])
    wide = {t: randn(g, n, 2 * pad_to(width, 8), dtype=t) for t in (dtype, torch.float32)}
    for terms in range(8):
        for yt in (dtype, torch.float32):
            log("sum_norm", width, dtype, terms, yt)
            y = wide[yt].to(DEV)[:, :width]
            u = wide[yt].to(DEV)[:, pad_to(width, 8):pad_to(width, 8) + width] if terms & 1 else None
            xd = x.to(DEV) if terms & 2 else None
            v = vec.to(DEV) if terms & 4 else None
            out, h = _mix.sum_norm(y, w.to(DEV), dtype, eps, x=xd, u=u, vec=v, mult=0.7, out=xd)
            want = 0.7 * y.cpu().double()
            want = want + (u.cpu().double() if terms & 1 else 0) + (x.double() if terms & 2 else 0) + (vec.double() if terms & 4 else 0)
            assert relative_rms(out, want) < 1e-6 and (terms & 2 == 0 or out is xd) and h.dtype == dtype
            assert relative_rms(h, S.rms(want, eps) * w.double()) < TOL[dtype]
    out, h = _mix.sum_norm(table.to(DEV), None, dtype, eps, tokens=tokens.to(DEV), mult=2.5)
    want = table[tokens].double() * 2.5
    assert relative_rms(out, want) < 1e-6 and relative_rms(h, want) < TOL[dtype]


@pytest.mark.parametrize("dtype", [BF16, torch.float32], ids=str)
@pytest.mark.parametrize("width", [100, 2048, 4096, 5000])
def test_a_row_s_norm_does_not_depend_on_how_many_there_are(width, dtype):
    """Weights loaded ahead of the reductions and behind them, at the lines between: the same bits."""
    g, rows = gen(width), 1281
    y, u = (randn(g, rows, width, dtype=dtype).to(DEV) for _ in range(2))
    x, w, v = randn(g, rows, width).to(DEV), randn(g, width).to(DEV), randn(g, width).to(DEV)

    def norms(n):
        planes, a, b = torch.stack([y[:n].float(), u[:n].float()]), x[:n].clone(), x[:n].clone()
        return (*_mix.sum_norm(y[:n], w, dtype, 1e-5, x=x[:n], u=u[:n], vec=v), _mix.residual_norm(y[:n], a, w, v, 0.5, 1e-5), a,
                *_mix.sum_norm(planes, w, dtype, 1e-5, x=x[:n]), _mix.residual_norm(planes, b, w, v, 0.5, 1e-5), b)

    few = norms(70)
    for n in (768, 769, 1024, 1025, 1280, 1281):
        log("rows", width, dtype, n)
        assert all(torch.equal(a, b[:70]) for a, b in zip(few, norms(n), strict=True))


@pytest.mark.parametrize("dtype", DTYPES)
def test_gelu_product(dtype):
    g = gen(5)
    for n, ff in ((1, 8), (5, 72), (300, 1000)):
        log("act_mul", n, ff, dtype)
        gu = randn(g, n, 2 * ff, dtype=dtype, std=3.0)
        want = S.gelu_tanh(gu[:, :ff].double()) * gu[:, ff:].double()
        assert relative_rms(_mix.act_mul(gu.to(DEV), "gelu_tanh"), want) < TOL[dtype]
    z = torch.tensor([[-1e4, -90.0, -8.0, 0.0, 8.0, 90.0, 1e4, 1.0] + [1.0] * 8]).to(dtype)
    y = _mix.act_mul(z.to(DEV), "gelu_tanh").cpu().float()
    assert torch.isfinite(y).all() and y[0, :3].abs().max() < 1e-9 and y[0, 6] == z[0, 6].float()


@pytest.mark.parametrize("dtype", DTYPES)
def test_norm_and_gate_of_each_head(dtype):
    g = gen(6)
    for n, heads, vp, count in ((1, 1, 32, 17), (9, 3, 96, 96), (5, 2, 288, 260), (130, 5, 64, 50)):
        log("head_gated_rms_norm", n, heads, vp, count, dtype)
        o = randn(g, n, heads, vp, dtype=dtype, std=5.0)
        o[..., count:] = 0
        gate, w = randn(g, n, heads * vp + 40, dtype=dtype), randn(g, vp) + 1
        got = _mix.head_gated_rms_norm(o.reshape(n, -1).to(DEV), gate.to(DEV)[:, 8:8 + heads * vp], w.to(DEV), count, 1e-2)
        want = S.rms(o[..., :count].double(), 1e-2) * w[:count].double()
        want = want * torch.sigmoid(gate[:, 8:8 + heads * vp].double().reshape(n, heads, vp)[..., :count])
        assert relative_rms(got.reshape(n, heads, vp)[..., :count].reshape(n, -1), want.reshape(n, -1)) < TOL[dtype]


# ---------------------------------------------------------------- grouped attention

# heads, kv_heads, dim, vdim: padding of either part, one head, no sharing, more rows than a tile, large heads
SHAPES = [(6, 3, 24, 40), (1, 1, 32, 32), (5, 5, 64, 96), (8, 2, 128, 128), (40, 2, 40, 16)]
LARGE = [(4, 2, 160, 128), (2, 1, 136, 200), (3, 1, 500, 64)]


class Attention:
    """Projected queries, keys, values and gates with padded head sizes, and a cache that a former sequence filled."""

    def __init__(self, shape, dtype, n, batch=1, seed=0, scale=None, softcap=0.0, sink=True, window=None, gate=True,
                 max_len=None):
        self.heads, self.groups, self.dim, self.vd = shape
        self.s = GqaShape(self.heads, self.groups, pad_to(self.dim), pad_to(self.vd), self.dim,
                          scale or self.dim ** -0.5, softcap, sink, _mix.UNBOUNDED if window is None else window)
        self.n, self.batch, self.dtype, self.gate = n, batch, dtype, gate
        g = gen(seed)
        self.q = randn(g, batch, n, self.heads, self.dim, dtype=dtype)
        self.k = randn(g, batch, n, self.groups, self.dim, dtype=dtype)
        self.v = randn(g, batch, n, self.groups, self.vd, dtype=dtype)
        self.z = randn(g, batch, n, self.heads, self.vd, dtype=dtype)
        self.max_len = max_len or n + 5
        self.cache = torch.full((batch, self.max_len, self.s.cache_cols), 7.0, dtype=dtype, device=DEV)

    def proj(self, lo, hi):
        s = self.s
        parts = [padded(t[:, lo:hi], p).reshape(self.batch * (hi - lo), -1)
                 for t, p in ((self.q, s.dk), (self.k, s.dk), (self.v, s.vp), (self.z, s.vp))]
        at = [0]
        for p in parts:
            at.append(at[-1] + p.size(1))
        return torch.cat(parts, 1).to(DEV), at

    def run(self, cuts, kind, nsplit=0, rot=None, norms=(None, None), eps=1e-5):
        """Portions of the given sizes through append and one of the three kernels."""
        out, lo, s = [], 0, self.s
        for c in cuts:
            proj, at = self.proj(lo, lo + c)
            pos = torch.arange(lo, lo + c, device=DEV)
            _mix.gqa_append(proj, s, at[1], at[2], rot, pos, *norms, self.cache, eps)
            g_off = at[3] if self.gate else -1
            if kind == "prefill":
                o = _mix.gqa_prefill(proj, s, g_off, self.cache, lo)
            else:
                o = _mix.gqa_rows(proj, s, g_off, self.cache, pos, kind == "rows", nsplit)
            out.append(o.cpu().reshape(self.batch, c, self.heads, s.vp))
            lo += c
        got = torch.cat(out, 1)
        assert got[..., self.vd:].count_nonzero() == 0
        return got[..., :self.vd].reshape(self.batch, self.n, -1)

    def want(self):
        rep, out = self.heads // self.groups, []
        d = torch.arange(self.n)[:, None] - torch.arange(self.n)[None]
        for b in range(self.batch):
            q, k, v = (t[b].double() for t in (self.q, self.k, self.v))
            o = torch.empty(self.n, self.heads, self.vd, dtype=torch.float64)
            for h in range(self.heads):
                x = q[:, h] @ k[:, h // rep].T * self.s.scale
                if self.s.softcap:
                    x = self.s.softcap * torch.tanh(x / self.s.softcap)
                x = x.masked_fill((d < 0) | (d >= self.s.window), float("-inf"))
                p = S.softmax_with_sink(x) if self.s.sink else torch.softmax(x, -1)
                o[:, h] = p @ v[:, h // rep]
            out.append(o * (torch.sigmoid(self.z[b].double()) if self.gate else 1))
        return torch.stack(out).reshape(self.batch, self.n, -1)


def kinds(dtype, shape):
    matrix = dtype == BF16 and max(shape[2:]) <= 128
    return ["general"] + ["rows"] * (dtype == BF16 and shape[2] <= 256 and shape[3] <= 128) + ["prefill"] * matrix


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
@pytest.mark.parametrize("shape", SHAPES + LARGE, ids=str)
def test_attention_of_portions(shape, dtype):
    for kind in kinds(dtype, shape):
        for i, cuts in enumerate(([150], [1, 2, 16, 31, 100], [130] + [1] * 10 + [5, 5])):
            if kind == "rows" and i == 0 and shape[0] > 30:
                continue
            log("attention", shape, dtype, kind, cuts[:4])
            c = Attention(shape, dtype, 150, batch=2, seed=i, softcap=(0.0, 2.0, 15.0)[i], sink=i != 1, gate=i != 2)
            err = max(relative_rms(a, b) for a, b in zip(c.run(cuts, kind), c.want()))
            assert err < TOL[dtype], err


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_one_far_key_is_found(dtype):
    """A query that points at one key among hundreds returns its value, wherever the key is: the first tokens, tile
    and split edges, the newest token."""
    shape, n = (4, 2, 64, 32), 521
    for kind in kinds(dtype, shape):
        for place in (0, 1, 31, 32, 63, 64, 127, 128, 255, 511, 519, 520):
            c = Attention(shape, dtype, n, seed=3, scale=1.0, softcap=25.0, gate=False)
            c.q *= 0.05
            c.q[0, 520, 3] = c.k[0, place, 1] / c.k[0, place, 1].float().pow(2).sum().sqrt() * 4
            c.k[0, place, 1] *= 8 / c.k[0, place, 1].float().pow(2).sum().sqrt() * 2
            for cuts, nsplit in (([n], 3), ([n - 1, 1], 5), ([500, 20, 1], 64)):
                if kind == "general" and nsplit != 5:
                    continue
                log("far key", dtype, kind, place, cuts, nsplit)
                got = c.run(cuts, kind, nsplit).reshape(n, 4, 32)
                # (25 tanh(64 / 25) = 24.7 against hundreds of scores near 0)
                assert relative_rms(got[520, 3], c.v[0, place, 1]) < 2 * TOL[BF16]
                assert relative_rms(got.reshape(n, -1), c.want()[0]) < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_the_sink_takes_what_no_key_wants(dtype):
    """Keys that point away from every query: with the sink the output all but vanishes, without it it is an
    average of the values."""
    shape, n = (2, 1, 32, 32), 140
    for kind in kinds(dtype, shape):
        for sink in (True, False):
            c = Attention(shape, dtype, n, seed=4, scale=1.0, softcap=12.0, sink=sink, gate=False)
            c.q[:] = 2.0
            c.k[:] = -2.0
            got = c.run([100, 7, 16, 16, 1], kind)
            log("sink", dtype, kind, sink, got.abs().max())
            # scores 12 tanh(-128 / 12) = -12: n e^-12 against 1
            assert relative_rms(got[0], c.want()[0]) < TOL[dtype]
            assert (got.abs().max() < 5e-3) == sink


@pytest.mark.parametrize("window", [1, 2, 33, 64, 129])
def test_attention_window_edges(window):
    for dtype in DTYPES:
        shape = (4, 2, 32, 32)
        for kind in kinds(dtype, shape):
            for cuts in ([300], [150] + [1] * 20 + [16, 114]):
                log("window", window, dtype, kind, cuts[:3])
                c = Attention(shape, dtype, 300, seed=window, window=window, softcap=8.0)
                c.k *= 3   # few keys carry the weight: one key too many or too few shows
                assert relative_rms(c.run(cuts, kind)[0], c.want()[0]) < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
@pytest.mark.parametrize("rot_dims", [2, 6, 16, 20, 40])
def test_append_norms_rotates_and_keeps_other_rows(rot_dims, dtype):
    shape, n, start, max_len, eps = (6, 2, 40, 72), 9, 30, 64, 1e-2
    log("append", rot_dims, dtype)
    c = Attention(shape, dtype, n, batch=2, max_len=max_len)
    g, s = gen(9), c.s
    wq, wk = randn(g, 40) + 1, randn(g, 40) + 1
    rot = Rotation(rot_dims, 300.0)
    proj, at = c.proj(0, n)
    pos = torch.arange(start, start + n)
    _mix.gqa_append(proj, s, at[1], at[2], rot.table(max_len).to(DEV), pos.to(DEV), padded(wq, s.dk).to(DEV),
                    padded(wk, s.dk).to(DEV), c.cache, eps)
    cache = c.cache.cpu().reshape(2, max_len, 2, s.dk + s.vp)
    untouched = torch.ones(max_len, dtype=torch.bool)
    untouched[start:start + n] = False
    assert cache[:, untouched].eq(7.0).all()
    rows, got_q = cache[:, start:start + n], proj.cpu()[:, :at[1]].reshape(2, n, 6, s.dk)
    for b in range(2):
        q = S.rotate_half(S.rms(c.q[b].double(), eps) * wq.double(), pos, rot_dims, 300.0)
        k = S.rotate_half(S.rms(c.k[b].double(), eps) * wk.double(), pos, rot_dims, 300.0)
        assert relative_rms(got_q[b, ..., :40].reshape(n, -1), q.reshape(n, -1)) < TOL[dtype]
        assert relative_rms(rows[b, ..., :40].reshape(n, -1), k.reshape(n, -1)) < TOL[dtype]
        assert torch.equal(rows[b, ..., s.dk:s.dk + 72], c.v[b]) and rows[b, ..., 40:s.dk].count_nonzero() == 0


# ---------------------------------------------------------------- short convolution


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 7])
def test_conv_in_portions(taps, dtype):
    g, batch, cols, n = gen(taps), 3, 44, 90
    x, w, bias = randn(g, batch, n, cols, dtype=dtype), randn(g, taps, cols), randn(g, cols)
    for silu in (False, True):
        want = [S.short_conv(x[b].double(), w.double().T) + (0 if silu else bias.double()) for b in range(batch)]
        want = [y * S.sigmoid(y) if silu else y for y in want]
        for cuts in ([n], [1] * n, [2] * 45, [9, 8, 3, 11, 19, 1, 2, 1, 36], [19, 19, 19, 19, 14]):
            log("conv", taps, dtype, silu, cuts[:4])
            ring = torch.full((batch, _mix.ring_rows(taps), cols), 50.0, dtype=dtype, device=DEV)   # a former sequence's
            out, lo = [], 0
            for c in cuts:
                proj = torch.zeros(batch * c, 72, dtype=dtype)
                proj[:, 20:20 + cols] = x[:, lo:lo + c].reshape(-1, cols)
                y = _mix.conv(proj.to(DEV), 20, w.to(DEV), None if silu else bias.to(DEV), ring,
                              torch.arange(lo, lo + c, device=DEV), silu)
                out.append(y.cpu().reshape(batch, c, cols))
                lo += c
            got = torch.cat(out, 1)
            assert max(relative_rms(got[b], want[b]) for b in range(batch)) < TOL[dtype]


# ---------------------------------------------------------------- gated linear recurrence


class Recurrence:
    def __init__(self, blocks, size, taps, dtype, n, batch=1, seed=0):
        g = gen(seed)
        self.blocks, self.size, self.taps, self.dtype, self.n, self.batch = blocks, size, taps, dtype, n, batch
        self.bp, c = pad_to(size), blocks * size
        self.x, self.y = randn(g, batch, n, c, dtype=dtype), randn(g, batch, n, c, dtype=dtype, std=2.0)
        self.wr, self.wi = (randn(g, blocks, size, size, dtype=dtype, std=size ** -0.5) for _ in range(2))
        # gates from shut to open: decays from a hair under 1 to none left
        self.br, self.bi = randn(g, c, std=3.0) - 2, randn(g, c)
        self.lam = torch.rand(c, generator=g) * 7 - 5
        self.cw, self.cb = randn(g, c, taps, std=taps ** -0.5), randn(g, c, std=0.2)
        self.state = torch.zeros(batch, blocks * self.bp, device=DEV)
        self.ring = torch.full((batch, _mix.ring_rows(taps), blocks * self.bp), 9.0, dtype=dtype, device=DEV)

    def pad(self, t):
        return padded(t.reshape(*t.shape[:-1], self.blocks, self.size), self.bp).reshape(*t.shape[:-1], -1)

    def run(self, cuts, kind, nseg=None):
        wr, wi = (padded(w, self.bp, self.bp).to(DEV) for w in (self.wr, self.wi))
        if kind == "general":
            wr, wi = wr.transpose(1, 2).contiguous(), wi.transpose(1, 2).contiguous()
        coef = (-8 * torch.nn.functional.softplus(self.lam.double())).float()
        gates = (wr, wi, self.pad(self.br).to(DEV), self.pad(self.bi).to(DEV), self.pad(coef).to(DEV), self.state)
        cw, cb = self.pad(self.cw.T.contiguous()).contiguous().to(DEV), self.pad(self.cb).to(DEV)
        out, lo, cols = [], 0, self.blocks * self.bp
        for c in cuts:
            proj = torch.cat([self.pad(t[:, lo:lo + c]).reshape(-1, cols) for t in (self.y, self.x)], 1).to(DEV)
            pos = torch.arange(lo, lo + c, device=DEV)
            if kind == "step":
                o = _mix.rglru_step(proj, 0, cols, cw, cb, self.ring, pos, *gates)
            else:
                u = _mix.conv(proj, cols, cw, cb, self.ring, pos, False)
                o = _mix.rglru(u, proj, 0, *gates, matrix=kind == "chunk",
                               nseg=None if nseg is None or kind != "chunk" else min(nseg, c))
            out.append(o.cpu().reshape(self.batch, c, self.blocks, self.bp)[..., :self.size])
            lo += c
        return torch.cat(out, 1).reshape(self.batch, self.n, -1)

    def want(self):
        outs, states = [], []
        for b in range(self.batch):
            u = S.short_conv(self.x[b].double(), self.cw.double()) + self.cb.double()
            if self.dtype == BF16:
                u = u.to(BF16).double()
            part = u.reshape(self.n, self.blocks, self.size)
            r, i = (torch.stack([S.sigmoid(part[:, k] @ w[k].double().T + bias.reshape(self.blocks, -1)[k].double())
                                 for k in range(self.blocks)], 1).reshape(self.n, -1)
                    for w, bias in ((self.wr, self.br), (self.wi, self.bi)))
            s, last = S.linear_unit_scan(u, r, i, self.lam.double())
            outs.append(s * S.gelu_tanh(self.y[b].double()))
            states.append(last)
        return outs, states

    def check(self, got, tol):
        outs, states = self.want()
        state = self.state.cpu().reshape(self.batch, self.blocks, self.bp)[..., :self.size].reshape(self.batch, -1)
        for b in range(self.batch):
            assert relative_rms(got[b], outs[b]) < tol
            assert relative_rms(state[b:b + 1], states[b][None]) < tol


# blocks x size: no padding, odd sizes, one block, several tiles per wave, the 64-token tile
BLOCKS = [(2, 32), (3, 30), (5, 8), (1, 100), (2, 256), (1, 330)]


@pytest.mark.parametrize("blocks,size", BLOCKS, ids=str)
@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_recurrence_in_portions(blocks, size, dtype):
    for kind in ["general"] + ["chunk"] * (dtype == BF16):
        for cuts in ([300], [129, 2, 1, 64, 104], [9, 127, 128, 36]):
            log("rglru", blocks, size, dtype, kind, cuts)
            c = Recurrence(blocks, size, 4, dtype, 300, batch=2, seed=size)
            c.check(c.run(cuts, kind), TOL[dtype])


@pytest.mark.parametrize("nseg", [1, 2, 3, 7])
def test_recurrence_in_segments(nseg):
    for size in (48, 300):
        log("rglru segments", nseg, size)
        c = Recurrence(2, size, 2, BF16, 1000, batch=2, seed=nseg)
        c.check(c.run([130, 870], "chunk", nseg), TOL[BF16])


@pytest.mark.parametrize("size", [64, 120, 192, 250])   # held weights: two, four, six and eight steps of 32 channels
@pytest.mark.parametrize("nseg", [1, 3])
def test_recurrence_held_weights(size, nseg):
    log("rglru held", nseg, size)
    c = Recurrence(3, size, 4, BF16, 400, batch=3, seed=size)
    c.check(c.run([63, 65, 193, 79] if nseg == 1 else [129, 271], "chunk", nseg), TOL[BF16])


@pytest.mark.parametrize("batch,taps", [(1, 4), (5, 3), (19, 2), (33, 1), (2, 7)])
def test_recurrence_step(batch, taps):
    for blocks, size in ((3, 30), (2, 256)):
        for cuts in ([1] * 24, [8, 8, 8], [5, 1, 3, 8, 2, 4, 1]):
            log("rglru step", batch, taps, size, cuts[:3])
            c = Recurrence(blocks, size, taps, BF16, 24, batch=batch, seed=batch)
            c.check(c.run(cuts, "step"), TOL[BF16])


def test_recurrence_at_the_ends_of_its_decay():
    """r all but 0: S grows like a sum whose terms shrink; r all but 1 and a large lam: nothing is kept."""
    for kind, dtype in (("general", torch.float32), ("general", BF16), ("chunk", BF16), ("step", BF16)):
        for br, lam in ((-12.0, -5.0), (12.0, 4.0)):
            c = Recurrence(1, 32, 4, dtype, 64, seed=2)
            c.wr *= 0
            c.br[:], c.lam[:] = br, lam
            log("decay ends", kind, dtype, br, lam)
            c.check(c.run([8] * 8, kind), TOL[dtype])


# ---------------------------------------------------------------- delta rule


class Delta:
    def __init__(self, shape, taps, dtype, n, batch=1, seed=0, z_std=2.0):
        self.heads, self.groups, self.dim, self.vd = shape
        h, k, d, v = shape
        g = gen(seed)
        self.s = DeltaShape(h, k, pad_to(d), pad_to(v), v, d ** -0.5)
        self.dtype, self.n, self.batch, self.taps = dtype, n, batch, taps
        self.q, self.k = (randn(g, batch, n, k, d, dtype=dtype) for _ in range(2))
        self.v = randn(g, batch, n, h, v, dtype=dtype)
        self.b = randn(g, batch, n, h, dtype=dtype, std=2.0)
        self.z = randn(g, batch, n, h, d, std=z_std)
        self.gate = randn(g, batch, n, h, v, dtype=dtype)
        self.dt, self.a_log = torch.rand(h, d, generator=g) * 5 - 4, torch.rand(h, generator=g) * 6 - 4.5
        self.norm = randn(g, v) * 0.3 + 1
        self.cw = [randn(g, c, taps, std=taps ** -0.5) for c in (k * d, k * d, h * v)]
        self.state = torch.zeros(batch, h, self.s.dp, self.s.vp, device=DEV)
        self.ring = torch.full((batch, _mix.ring_rows(taps), self.s.qkv_cols), 9.0, dtype=dtype, device=DEV)
        self.eps = 1e-3

    def run(self, cuts, kind):
        s, out, lo = self.s, [], 0
        cw = torch.cat([padded(w.reshape(-1, p, self.taps), q, self.taps).reshape(-1, self.taps)
                        for w, p, q in zip(self.cw, (self.dim, self.dim, self.vd), (s.dp, s.dp, s.vp))]).T.contiguous().to(DEV)
        dt, decay, norm = padded(self.dt, s.dp).reshape(-1).to(DEV), self.a_log.double().exp().float().to(DEV), padded(self.norm, s.vp).to(DEV)
        for c in cuts:
            def rows(t, p):
                return padded(t[:, lo:lo + c], p).reshape(self.batch * c, -1)
            proj = torch.cat([rows(self.q, s.dp), rows(self.k, s.dp), rows(self.v, s.vp), rows(self.b, pad_to(self.heads, 8))], 1).to(DEV)
            z, gate = rows(self.z, s.dp).to(DEV), rows(self.gate, s.vp).to(DEV)
            pos, rule = torch.arange(lo, lo + c, device=DEV), (s, s.qkv_cols, z, dt, decay)
            if kind == "fused":
                o = _mix.delta_step(proj, *rule, gate, norm, self.state, self.eps, x_off=0, conv_w=cw, ring=self.ring, positions=pos)
            else:
                qkv = _mix.conv(proj, 0, cw, None, self.ring, pos, True)
                if kind == "step":
                    o = _mix.delta_step(proj, *rule, gate, norm, self.state, self.eps, qkv=qkv)
                else:
                    o = _mix.delta_chunk(qkv, proj, *rule, self.state)
                    o = _mix.head_gated_rms_norm(o, gate, norm, self.vd, self.eps)
            out.append(o.cpu().reshape(self.batch, c, self.heads, s.vp))
            lo += c
        got = torch.cat(out, 1)
        assert got[..., self.vd:].count_nonzero() == 0
        return got[..., :self.vd].reshape(self.batch, self.n, -1)

    def want(self, conv=True):
        rep, outs, states = self.heads // self.groups, [], []
        for b in range(self.batch):
            def mixed(t, w):
                y = S.short_conv(t[b].double().reshape(self.n, -1), w.double())
                y = y * S.sigmoid(y)
                return (y.to(BF16).double() if self.dtype == BF16 else y).reshape(t[b].shape)
            q, k, v = mixed(self.q, self.cw[0]), mixed(self.k, self.cw[1]), mixed(self.v, self.cw[2])
            q, k = S.unit(q) * self.dim ** -0.5, S.unit(k)
            g = torch.exp(-self.a_log.double().exp()[:, None] * S.softplus(self.z[b].double() + self.dt.double()))
            o, s = S.delta_scan(q.repeat_interleave(rep, 1), k.repeat_interleave(rep, 1), v, g, S.sigmoid(self.b[b].double()))
            outs.append((S.rms(o, self.eps) * self.norm.double() * S.sigmoid(self.gate[b].double())).reshape(self.n, -1))
            states.append(s)
        return outs, states

    def errors(self, got):
        """(of the output, of the state) of each sequence."""
        outs, states = self.want()
        state = self.state.cpu()[:, :, :self.dim, :self.vd]
        return [(relative_rms(got[b], outs[b]), relative_rms(state[b].reshape(1, -1), states[b].reshape(1, -1))) for b in range(self.batch)]

    def check(self, got, tol):
        for err in self.errors(got):
            # (the state has no bf16 in it but its inputs)
            assert err[0] < tol and err[1] < (tol if tol < 1e-4 else 1e-4), err


DELTAS = [(4, 2, 40, 24), (1, 1, 32, 32), (3, 3, 64, 96), (2, 1, 128, 128), (2, 2, 100, 136), (2, 1, 160, 64), (1, 1, 256, 256)]


@pytest.mark.parametrize("shape", DELTAS, ids=str)
@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_delta_rule_in_portions(shape, dtype):
    for kind in ["step"] + ["chunk"] * (dtype == BF16):
        for cuts in ([120], [33, 2, 1, 16, 17, 15, 36], [9, 64, 47]):
            log("delta", shape, dtype, kind, cuts)
            c = Delta(shape, 3, dtype, 120, batch=2, seed=shape[2])
            c.check(c.run(cuts, kind), TOL[dtype])


@pytest.mark.parametrize("batch,taps", [(1, 4), (3, 2), (2, 1), (2, 7)])
@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_delta_rule_fused_step(batch, taps, dtype):
    for shape in ((4, 2, 40, 24), (2, 1, 128, 128), (2, 2, 64, 200)):
        for cuts in ([1] * 24, [8, 8, 8], [5, 1, 3, 8, 2, 4, 1]):
            log("delta fused", batch, taps, shape, dtype, cuts[:3])
            c = Delta(shape, taps, dtype, 24, batch=batch, seed=batch)
            c.check(c.run(cuts, "fused"), TOL[dtype])


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_delta_rule_under_strong_decays(dtype):
    """Decays of e^-50 and more per token beside channels that keep everything: a chunk's products over- and underflow
    unless every factor is at most 1."""
    for kind in ["step"] + ["chunk"] * (dtype == BF16):
        c = Delta((2, 1, 64, 64), 2, dtype, 80, seed=8, z_std=1.0)
        c.z[..., ::3] = 60.0
        c.z[..., 1::3] = -60.0
        c.z[:, 20:24] = 30.0
        c.a_log[:] = 0.5
        log("strong decays", kind, dtype)
        c.check(c.run([50, 30], kind), TOL[dtype])


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16"])
def test_delta_rule_with_equal_keys(dtype):
    """One key over and over with beta near 1 and no decay: every write takes the one before it off, the
    chunk's triangular system is as full as it gets."""
    for kind in ["step"] + ["chunk"] * (dtype == BF16):
        c = Delta((2, 2, 32, 32), 1, dtype, 70, seed=9)
        c.k[:] = c.k[:, :1]
        c.b[:], c.z[:] = 6.0, -30.0
        c.a_log[:] = -6.0
        log("equal keys", kind, dtype)
        c.check(c.run([40, 30], kind), TOL[dtype])


@pytest.mark.parametrize("shape", DELTAS + [(9, 3, 32, 64)], ids=str)
def test_delta_rule_in_blocks(shape, monkeypatch):
    """Blocks of 64 tokens whatever the size: at their edges, under decays whose products over- and underflow, and with one
    key over and over. Beside chunks of 16, on the same inputs: a convolved input whose bf16 rounding falls the other way than
    the oracle's is 2^-9 of it in both (seed 129: 1.8e-4 of the state), so that far a state may be off besides its own 1e-4. (80 equal
    keys: what their writes leave is a difference of rounded inputs, 1.3e-2 of the output after 150 in chunks of 16 alike.)"""
    for cuts in ([1, 63, 64, 65], [16, 17, 128, 129], [33, 191]):
        for seed in (shape[2] + 1, shape[2] + 2):
            errors = []
            for blocks in (False, True):
                log("delta blocks", shape, cuts, seed, blocks)
                monkeypatch.setattr(_mix, "delta_in_blocks", lambda *a: blocks)
                c = Delta(shape, 3, BF16, sum(cuts), batch=2, seed=seed)
                errors.append(c.errors(c.run(cuts, "chunk")))
            for chunks, err in zip(*errors):
                assert err[0] < TOL[BF16] and err[1] < 1e-4 + chunks[1], (chunks, err)
    c = Delta(shape, 2, BF16, 144, seed=8, z_std=1.0)
    c.z[..., ::3] = 60.0
    c.z[..., 1::3] = -60.0
    c.z[:, 20:24] = 30.0
    c.a_log[:] = 0.5
    c.check(c.run([100, 44], "chunk"), TOL[BF16])
    c = Delta(shape, 1, BF16, 80, seed=9)
    c.k[:] = c.k[:, :1]
    c.b[:], c.z[:] = 6.0, -30.0
    c.a_log[:] = -6.0
    c.check(c.run([66, 14], "chunk"), TOL[BF16])


@pytest.mark.parametrize("bad", [float("nan"), float("inf")], ids=str)
@pytest.mark.parametrize("what", ["q", "k", "v", "z", "b"])
def test_delta_rule_in_blocks_keeps_what_is_not_finite_from_earlier_tokens(what, bad, monkeypatch):
    """A token's NaN or infinity reaches the same outputs and states as in chunks of 16: none before its 16."""
    s, n = DeltaShape(3, 3, 64, 64, 64, 0.125), 150
    for token in (0, 16, 31, 40, 63, 64, 149):
        g, seen = gen(token), []
        proj, z = randn(g, n, s.qkv_cols + 8, dtype=BF16), randn(g, n, 3 * 64)
        if what == "z":
            z[token, 3] = bad
        else:
            proj[token, {"q": 3, "k": 3 * 64 + 3, "v": 6 * 64 + 3, "b": s.qkv_cols}[what]] = bad
        qkv, proj, z = proj[:, :s.qkv_cols].contiguous().to(DEV), proj.to(DEV), z.to(DEV)
        for blocks in (False, True):
            log("delta not finite", what, bad, token, blocks)
            state = torch.ones(1, 3, 64, 64, device=DEV)
            monkeypatch.setattr(_mix, "delta_in_blocks", lambda *a: blocks)
            out = _mix.delta_chunk(qkv, proj, s, s.qkv_cols, z, torch.zeros(3 * 64, device=DEV), torch.ones(3, device=DEV), state)
            seen.append((out.isfinite(), state.isfinite()))
        assert all(torch.equal(a, b) for a, b in zip(*seen))
        assert seen[1][0][:token // 16 * 16].all()


@pytest.mark.parametrize("batch,seq,cut", [(1, 16400, 129 * 64), (2, 8300, 65 * 64)])
def test_delta_rule_in_blocks_of_a_prompt_in_parts(batch, seq, cut):
    """Operands of more than 512 MiB are formed and walked in two parts: the bits of a call for each, at a block's edge."""
    s = DeltaShape(16, 16, 128, 128, 128, 0.09)
    size = _mix._require().astrai_mix_delta_blocks_bytes
    assert size(batch, 16, seq, 128, 128) == size(batch, 16, cut, 128, 128) < size(batch, 16, cut + 64, 128, 128)
    torch.manual_seed(seq)
    mk = lambda cols, dtype=BF16: torch.randn(batch, seq, cols, device=DEV).to(dtype)
    qkv, proj, z, dt, decay = mk(s.qkv_cols), mk(s.qkv_cols + 16), mk(16 * 128, torch.float32), torch.zeros(16 * 128, device=DEV), torch.ones(16, device=DEV)
    got = []
    for cuts in ([(0, seq)], [(0, cut), (cut, seq)]):
        state, outs = torch.ones(batch, 16, 128, 128, device=DEV), []
        for a, b in cuts:
            log("delta parts", batch, a, b)
            part = [t[:, a:b].reshape(batch * (b - a), -1).contiguous() for t in (qkv, proj, z)]
            outs.append(_mix.delta_chunk(part[0], part[1], s, s.qkv_cols, part[2], dt, decay, state, blocks=True).view(batch, b - a, -1))
        got.append((torch.cat(outs, 1), state))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and got[0][0].isfinite().all()


def test_delta_rule_in_blocks_where_they_are_taken():
    shape = (2, 1, 64, 64)
    for batch, n in ((1, 768), (2, 1030)):
        assert _mix.delta_in_blocks(batch, n, DeltaShape(2, 1, 64, 64, 64, 0.125))
        c = Delta(shape, 3, BF16, n, batch=batch, seed=11)
        c.check(c.run([n], "chunk"), TOL[BF16])


def test_a_write_far_back_is_read():
    """One strong write whose key no later key touches, decays all but 1: its value comes back hundreds of tokens
    later, through chunks and steps alike."""
    n = 600
    for kind, dtype, cuts in (("step", torch.float32, [n]), ("chunk", BF16, [n]), ("chunk", BF16, [17] * 35 + [5]), ("fused", BF16, [8] * 75)):
        c = Delta((1, 1, 32, 32), 1, dtype, n, seed=10)
        for w in c.cw:
            w[:] = 1.0
        c.k[..., 0], c.q[..., 0] = -30.0, -30.0     # (silu takes the channel out)
        c.k[0, 5], c.k[0, 5, :, 0] = -30.0, 8.0
        c.b[0, 5], c.z[:] = 9.0, -40.0
        c.q[0, n - 1], c.q[0, n - 1, :, 0] = -30.0, 8.0
        log("far write", kind, dtype)
        got = c.run(cuts, kind)
        c.check(got, TOL[dtype])
        v = c.v[0, 5, 0].double()
        v = v * S.sigmoid(v)
        state = c.state.cpu()[0, 0, 0, :32]
        assert relative_rms(state[None], v[None]) < 2e-2


def test_wrong_operands_are_refused_before_a_launch():
    s = GqaShape(2, 1, 32, 32, 32, 0.2)
    proj, cache = torch.zeros(4, 192, device=DEV), torch.zeros(1, 8, 64, device=DEV)
    pos = torch.arange(4, device=DEV)
    with pytest.raises(RuntimeError, match="cache rows"):
        _mix.gqa_rows(proj, s, -1, torch.zeros(1, 8, 96, device=DEV), pos, False)
    with pytest.raises(RuntimeError, match="expected shape"):
        _mix.gqa_append(proj, s, 64, 96, None, pos[:3], None, None, cache, 1e-6)
    with pytest.raises(RuntimeError, match="bf16|expected torch.bfloat16"):
        _mix.gqa_prefill(proj, s, -1, cache, 0)
    with pytest.raises(RuntimeError, match="ring"):
        _mix.conv(proj, 0, torch.zeros(3, 64, device=DEV), None, torch.zeros(1, 9, 64, device=DEV), pos, False)
    with pytest.raises(RuntimeError, match="GPU required"):
        _mix.sum_norm(torch.zeros(2, 16), None, torch.float32, 1e-6)
