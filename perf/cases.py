"""What a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values; its ``kind`` says which entry point it goes through:

  ``linear_int8``  ``F.linear`` under ``int8_autocast``: weights quantized once, tokens on every call
  ``linear_fp8``   ``F.linear`` under ``fp8_autocast`` without gradients, delayed or dynamic scaling
  ``train_fp8``    the same with gradients: output, input, weight and bias gradient of one step
  ``linear_block`` 128-block fp8: activations quantized on every call, then the block-scaled product
  ``prompt_attn``  attention of a block of new tokens, dense tensors (``[batch, seq, heads, dim]``) or a
                   ragged batch over a pool of cached rows behind a slot table
  ``decode_attn``  attention of one new token per sequence over such a pool
  ``prompt``       a model's forward over a prompt, with the logits that the next token is chosen from
  ``step``         a model's decode step, captured once and replayed as the generation loop replays it

Every function takes the case; inputs are made on the GPU from the seed alone.
"""

import math

import torch
import torch.nn.functional as F

from astrai_amd.extension import _cabi, fp8, w8a8
from astrai_amd.extension.ops import attention as attn_ops
from astrai_amd.extension.ops import fp8_block
from astrai_amd.model import (AutoRegressiveLM, AutoRegressiveLMConfig, LugitarConfig, LugitarLM, SarulixConfig,
                              SarulixLM, fuse_int8_weights)

DEV = "cuda"
VOCAB = 32000
# (inner size, outputs) of the projections of the configured decoders: q|k|v, output, gate|up, down, head
PROJECTIONS = [(2048, 2048), (2048, 3072), (2048, 11264), (5632, 2048), (4096, 4096), (4096, 11008), (11008, 4096)]
BLOCK_PROJECTIONS = [(7168, 2048), (2048, 7168), (4096, 4096), (7168, 1536)]
# (query heads, key/value heads, head size)
HEADS = [(16, 4, 128), (32, 8, 128), (32, 8, 64), (16, 16, 64), (16, 16, 128), (32, 4, 128)]


def listed():
    return [
        # one projection of a serving batch's decode step outside a captured graph: 45 MB of weights
        dict(name="int8 linear 16 tokens", kind="linear_int8", tokens=16, k=4096, n=11008, bias=False),
        # a prompt whose length is no multiple of anything, through a feed-forward projection with a bias
        dict(name="fp8 linear 3001 tokens", kind="linear_fp8", tokens=3001, k=2048, n=11264, bias=True, dynamic=True),
        # one training step's linear layer, forward and backward
        dict(name="fp8 training 4096", kind="train_fp8", tokens=4096, k=4096, n=4096, bias=True, dynamic=False),
        # the block-scaled product of a large prompt
        dict(name="block fp8 8192 tokens", kind="linear_block", tokens=8192, k=7168, n=2048),
        # causal attention of fresh prompts, tensors as the model's projections give them
        dict(name="prompt attention dense", kind="prompt_attn", paged=False, batch=4, new=2048, cached=0, heads=16,
             kv_heads=4, dim=128),
        # a ragged batch of a paged server, some of each prompt's prefix cached already, heads of 64
        dict(name="prompt attention paged", kind="prompt_attn", paged=True, batch=16, new=700, cached=500, heads=32,
             kv_heads=8, dim=64),
        # a paged server's decode step, ragged contexts
        dict(name="decode attention paged", kind="decode_attn", batch=32, context=3000, heads=16, kv_heads=4, dim=128),
        # a batch of prompts through the dense decoder, int8 weights and activations
        dict(name="dense int8 prompt 32 x 512", kind="prompt", model="dense", batch=32, seq=512),
        # ... and the decode step that follows
        dict(name="dense int8 step 32 x 512", kind="step", model="dense", batch=32, seq=512),
        # a batch of prompts through latent and lightning attention
        dict(name="lugitar prompt 32 x 512", kind="prompt", model="lugitar", batch=32, seq=512),
        # one long prompt through recurrences, delta rule and attention with a sink
        dict(name="sarulix prompt 1 x 4096", kind="prompt", model="sarulix", batch=1, seq=4096),
        # ... and a batch's decode step
        dict(name="sarulix step 32 x 512", kind="step", model="sarulix", batch=32, seq=512),
    ]


def draw(rng):
    def spread(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["linear_int8", "linear_fp8", "train_fp8", "linear_block", "prompt_attn", "prompt_attn",
                       "decode_attn", "prompt", "step"])
    case = dict(kind=kind)
    if kind == "linear_block":
        k, n = rng.choice(BLOCK_PROJECTIONS)
        case.update(tokens=spread(4, 8192), k=k, n=n)
    elif kind in ("linear_int8", "linear_fp8", "train_fp8"):
        k, n = rng.choice(PROJECTIONS)
        case.update(tokens=spread(1, 4096) if kind != "train_fp8" else spread(256, 2500), k=k, n=n,
                    bias=rng.random() < 0.5)
        if kind != "linear_int8":
            case["dynamic"] = rng.random() < 0.5
    elif kind == "prompt_attn":
        heads, kv_heads, dim = rng.choice(HEADS)
        paged = rng.random() < 0.5
        batch, new = spread(1, 32), spread(33, 4096)
        cached = spread(1, 2048) if paged and rng.random() < 0.7 else 0
        while batch > 1 and batch * heads * dim * new * (new + 2 * cached) > 5e11:
            batch -= 1
        case.update(paged=paged, batch=batch, new=new, cached=cached, heads=heads, kv_heads=kv_heads, dim=dim)
    elif kind == "decode_attn":
        heads, kv_heads, dim = rng.choice(HEADS)
        batch, context = spread(1, 128), spread(64, 8192)
        while batch > 1 and batch * context > 131072:
            batch -= 1
        case.update(batch=batch, context=context, heads=heads, kv_heads=kv_heads, dim=dim)
    else:
        batch = spread(1, 32)
        case.update(model=rng.choice(["dense", "lugitar", "sarulix"]), batch=batch,
                    seq=spread(32, min(4096, 8192 // batch)))
    return case


# ---- inputs --------------------------------------------------------------------------------------------------

class _Random:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *size, std=1.0, mean=0.0):
        return (torch.randn(*size, generator=self.g, device=DEV) * std + mean).to(torch.bfloat16)

    def uniform(self, lo, hi, *size):
        return (torch.rand(*size, generator=self.g, device=DEV) * (hi - lo) + lo).to(torch.bfloat16)

    def ints(self, hi, *size):
        return torch.randint(0, hi, size, generator=self.g, device=DEV)

    def order(self, n):
        return torch.randperm(n, generator=self.g, device=DEV)


def _linear_inputs(case, seed):
    r = _Random(seed)
    x = r.normal(case["tokens"], case["k"])
    w = r.normal(case["n"], case["k"], std=0.02)
    b = r.normal(case["n"], std=0.1) if case.get("bias") else None
    g = r.normal(case["tokens"], case["n"], std=0.01) if case["kind"] == "train_fp8" else None
    return x, w, b, g


def _lengths(case):
    """Ragged lengths around the case's: what each sequence of a batch holds."""
    n = case["batch"]
    share = [1.0 - 0.75 * ((5 * i) % n) / n for i in range(n)]
    return share


def _prompt_attn_inputs(case, seed):
    r, b, d = _Random(seed), case["batch"], case["dim"]
    h, g = case["heads"], case["kv_heads"]
    if not case["paged"]:
        n = case["new"]
        return dict(q=r.normal(b, n, h, d), k=r.normal(b, n, g, d), v=r.normal(b, n, g, d))
    share = _lengths(case)
    new = [max(1, int(case["new"] * s)) for s in share]
    kv = [n + int(case["cached"] * s) for n, s in zip(new, reversed(share))]
    slots, most = sum(kv) + 64, max(kv)
    order = r.order(slots).int()
    table = torch.full((b, most), -1, device=DEV, dtype=torch.int32)
    at = 0
    for i, n in enumerate(kv):
        table[i, :n] = order[at:at + n]
        at += n
    return dict(q=r.normal(sum(new), h, d), k=r.normal(slots, g, d), v=r.normal(slots, g, d), table=table, new=new,
                kv=kv)


def _decode_attn_inputs(case, seed):
    r, b, d = _Random(seed), case["batch"], case["dim"]
    kv = [max(1, int(case["context"] * s)) for s in _lengths(case)]
    slots, most = sum(kv) + 64, max(kv)
    order = r.order(slots).int()
    table = torch.full((b, most), -1, device=DEV, dtype=torch.int32)
    at = 0
    for i, n in enumerate(kv):
        table[i, :n] = order[at:at + n]
        at += n
    return dict(q=r.normal(b, case["heads"], d), k=r.normal(slots, case["kv_heads"], d),
                v=r.normal(slots, case["kv_heads"], d), table=table, kv=kv)


def _starts(lengths):
    out = [0]
    for n in lengths:
        out.append(out[-1] + n)
    return out


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


# ---- models: a few layers of each design at the sizes of the configured decoders -------------------------------
# (two of the dense decoder: a rounding that falls the other way re-rounds int8 codes in every layer behind it)

WIDTH, HEAD_COUNT, FF, LAYERS = 2048, 16, 5632, 2


def _config(name):
    if name == "dense":
        return dict(hidden_size=WIDTH, num_hidden_layers=LAYERS, num_attention_heads=HEAD_COUNT,
                    num_key_value_heads=HEAD_COUNT // 4, intermediate_size=FF, vocab_size=VOCAB,
                    max_position_embeddings=4224)
    mlp = {"kind": "dense", "ff": FF}
    if name == "lugitar":
        rot = {"dims": 64, "base": 10000.0, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}
        latent = {"heads": HEAD_COUNT, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "rot": rot,
                  "scale": 192 ** -0.5, "mask": {"size": 1024}}
        decay = [1.0 - 2.0 ** (-2 - 6 * i / HEAD_COUNT) for i in range(HEAD_COUNT)]
        lightning = {"heads": HEAD_COUNT, "dim": 128, "vdim": 128, "decay": decay}
        layers = [("latent_attention", latent), ("lightning", lightning),
                  ("latent_attention", {**latent, "kv_from": 0}), ("lightning", lightning)]
        return {"architecture": "Lugitar", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-5}, "residual_mult": 0.5,
                "layers": [{"type": t, "mixer": m, "mlp": mlp} for t, m in layers]}
    rglru = {"width": WIDTH, "blocks": WIDTH // 256, "conv": 4}
    delta = {"heads": HEAD_COUNT, "kv_heads": HEAD_COUNT, "dim": 128, "vdim": 128, "conv": 4}
    attention = {"heads": HEAD_COUNT, "kv_heads": HEAD_COUNT // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                 "softcap": 50.0, "rot": {"dims": 64, "base": 10000.0}}
    layers = [("rglru", rglru), ("channel_delta", delta), ("rglru", rglru), ("attention", attention)]
    return {"architecture": "Sarulix", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-5},
            "embedding": {"scale": 1.0}, "logit_scale": 1.0, "loop": {"start": 1, "stop": 3, "times": 2},
            "layers": [{"type": t, "mixer": m, "mlp": mlp} for t, m in layers]}


def _weights(name, seed):
    """Tensors by the names under which a checkpoint stores them."""
    r, cfg, out = _Random(seed), _config(name), {}

    def matrix(key, rows, cols):
        out[key] = r.normal(rows, cols, std=cols ** -0.5)

    if name == "dense":
        d, kv = WIDTH, cfg["num_key_value_heads"] * WIDTH // HEAD_COUNT
        out["embed_tokens.weight"] = r.normal(VOCAB, d)
        for i in range(LAYERS):
            p = f"layers.{i}."
            for key, rows, cols in (("attention.q_proj", d, d), ("attention.k_proj", kv, d), ("attention.v_proj", kv, d),
                                    ("attention.o_proj", d, d), ("mlp.gate", FF, d), ("mlp.up", FF, d), ("mlp.down", d, FF)):
                matrix(p + key + ".weight", rows, cols)
            out[p + "input_norm.weight"] = r.normal(d, std=0.1, mean=1.0)
            out[p + "post_attention_norm.weight"] = r.normal(d, std=0.1, mean=1.0)
        out["norm.weight"] = r.normal(d, std=0.1, mean=1.0)
        matrix("lm_head.weight", VOCAB, d)
        return out
    w, around = cfg["width"], 1.0 if name == "lugitar" else 0.0
    out["embed"] = r.normal(VOCAB, w)
    if "loop" in cfg:
        matrix("loop.in", w, 2 * w)
        out["loop.step"] = r.normal(cfg["loop"]["times"], w, std=0.3)
    for i, layer in enumerate(cfg["layers"]):
        p, m = f"l{i}.mix.", layer["mixer"]
        for norm in ("norm1", "norm2") + (("norm1b", "norm2b") if name == "lugitar" else ()):
            out[f"l{i}.{norm}"] = r.normal(w, std=0.1, mean=around)
        h, d, v = m.get("heads"), m.get("dim"), m.get("vdim")
        if layer["type"] == "latent_attention":
            matrix(p + "q", h * (d + m["rot_dim"]), w)
            if "kv_from" not in m:
                matrix(p + "dkv", m["kv_rank"] + m["rot_dim"], w)
                out[p + "dkv.norm"] = r.normal(m["kv_rank"], std=0.1, mean=1.0)
            matrix(p + "uk", h * d, m["kv_rank"])
            matrix(p + "uv", h * v, m["kv_rank"])
            matrix(p + "g", h, w)
        elif layer["type"] == "lightning":
            for key in ("q", "k", "v", "g"):
                matrix(p + key, h * d, w)
            out[p + "norm"] = r.normal(h * v, std=0.1, mean=1.0)
        elif layer["type"] == "attention":
            for key, n in (("q", h * d), ("k", m["kv_heads"] * d), ("v", m["kv_heads"] * v)):
                matrix(p + key, n, w)
                out[p + key + ".b"] = r.normal(n, std=0.1)
            matrix(p + "g", h * v, w)
            out[p + "q.norm"], out[p + "k.norm"] = r.normal(d, std=0.1, mean=1.0), r.normal(d, std=0.1, mean=1.0)
            out[p + "o.b"] = r.normal(w, std=0.1)
        elif layer["type"] == "rglru":
            c, b = m["width"], m["blocks"]
            for key in ("y", "x"):
                matrix(p + key, c, w)
                out[p + key + ".b"] = r.normal(c, std=0.1)
            out[p + "conv"], out[p + "conv.b"] = r.normal(c, m["conv"], std=m["conv"] ** -0.5), r.normal(c, std=0.1)
            for key in ("ra", "ri"):
                out[p + key] = r.normal(b, c // b, c // b, std=(c // b) ** -0.5)
                out[p + key + ".b"] = r.normal(b, c // b)
            out[p + "lam"] = r.uniform(-5, 0, c)
        else:
            for key in ("q", "k", "v"):
                matrix(p + key, h * d, w)
                out[p + key + ".conv"] = r.normal(h * d, m["conv"], std=m["conv"] ** -0.5)
            matrix(p + "b", h, w)
            out[p + "A_log"], out[p + "dt_bias"] = r.uniform(-2, 1, h), r.uniform(-5, 0, h * d)
            for low, high in (("a1", "a2"), ("g1", "g2")):
                matrix(p + low, v, w)
                matrix(p + high, h * d, v)
            out[p + "norm"] = r.normal(v, std=0.1, mean=1.0)
        matrix(p + "o", w, h * v if h else m["width"])
        matrix(f"l{i}.mlp.gate", FF, w)
        matrix(f"l{i}.mlp.up", FF, w)
        matrix(f"l{i}.mlp.down", w, FF)
    out["final.norm"] = r.normal(w, std=0.1, mean=around)
    matrix("head", VOCAB, w)
    return out


def _model(name, weights):
    cfg = _config(name)
    with torch.device(DEV):
        if name == "dense":
            model = AutoRegressiveLM(AutoRegressiveLMConfig(**cfg))
        elif name == "lugitar":
            model = LugitarLM(LugitarConfig.from_dict(cfg))
        else:
            model = SarulixLM(SarulixConfig.from_dict(cfg).with_tensors(weights))
    model = model.to(torch.bfloat16).eval().load_tensors(weights)
    if name == "dense":
        fuse_int8_weights(model)
    return model


def _prompt_ids(case, seed, extra=0):
    return _Random(seed + 1_000_003).ints(VOCAB, case["batch"], case["seq"] + extra)


def _held(cache):
    """What a cache carries on to the next token."""
    if hasattr(cache, "state"):
        return {"state": list(cache.state.values()), "rows": list(cache.rows.values())}
    return {"rows": [cache.k, cache.v]}


# ---- a case's state and one pass ---------------------------------------------------------------------------------

@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("linear_int8", "linear_fp8", "train_fp8", "linear_block"):
        x, w, b, g = _linear_inputs(case, seed)
        s = dict(case=case, x=x, w=w, b=b, g=g)
        if kind == "linear_int8":
            w8a8.int8_state().get_weight(w)            # weights are quantized when a model is loaded
        elif kind == "linear_block":
            s["w8"], s["sw"] = fp8_block.quantize_weight_block128(w)
        else:
            fp8.fp8_state().reset()                    # another model's scaling state is no part of this one's
            s["recipe"] = fp8.DynamicScaling() if case["dynamic"] else fp8.DelayedScaling()
            if kind == "train_fp8":
                for t in (x, w, b):
                    if t is not None:
                        t.requires_grad_(True)
        return s
    if kind == "prompt_attn":
        s = _prompt_attn_inputs(case, seed)
        if case["paged"]:
            s["rows"], s["kv_indptr"] = _int32(list(range(case["batch"]))), _int32(_starts(s["kv"]))
            s["schedule"] = _cabi.paged_prefill_schedule(s["new"], DEV)
        return dict(case=case, **s)
    if kind == "decode_attn":
        s = _decode_attn_inputs(case, seed)
        return dict(case=case, rows=_int32(list(range(case["batch"]))), kv_indptr=_int32(_starts(s["kv"])), **s)
    model = _model(case["model"], _weights(case["model"], seed))
    batch, seq = case["batch"], case["seq"]
    ids, cache = _prompt_ids(case, seed, 1), model.new_cache(batch, seq + 64)
    s = dict(case=case, model=model, cache=cache, ids=ids[:, :seq].contiguous(),
             last=torch.tensor([seq - 1], device=DEV))
    if kind == "prompt":
        return s
    # the generation loop: prompt, one eager step, capture; a replay reads the token and its place from these
    # buffers and runs the step at the same place every time
    s["token"], s["place"] = ids[:, seq:].contiguous(), torch.tensor([seq], device=DEV)
    with w8a8.int8_autocast(case["model"] == "dense"):
        for _ in range(2):
            cache.reset()
            model(s["ids"], cache, logits_at=s["last"])
            cache.advance(seq)
            if "graph" not in s:
                model(s["token"], cache, s["place"])
                s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["logits"] = model(s["token"], cache, s["place"])["logits"]
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear_int8":
        with torch.no_grad(), w8a8.int8_autocast(True):
            return F.linear(s["x"], s["w"], s["b"])
    if kind == "linear_fp8":
        with torch.no_grad(), fp8.fp8_autocast(True, recipe=s["recipe"]):
            return F.linear(s["x"], s["w"], s["b"])
    if kind == "train_fp8":
        with fp8.fp8_autocast(True, recipe=s["recipe"]):
            out = F.linear(s["x"], s["w"], s["b"])
            leaves = [t for t in (s["x"], s["w"], s["b"]) if t is not None]
            return {"out": out.detach(), "grads": torch.autograd.grad(out, leaves, s["g"])}
    if kind == "linear_block":
        x8, sx = fp8_block.quantize_act_block128(s["x"])
        return fp8_block.mm_fp8_blockscaled(x8, s["w8"], sx, s["sw"])
    if kind == "prompt_attn":
        if not case["paged"]:
            return attn_ops.attn_prefill(s["q"], s["k"], s["v"], is_causal=True)
        return attn_ops.attn_paged_prefill(s["q"], s["k"], s["v"], s["table"], s["rows"], s["kv_indptr"], *s["schedule"],
                                           is_causal=True)
    if kind == "decode_attn":
        return attn_ops.attn_paged_decode(s["q"], s["k"], s["v"], s["table"], s["rows"], s["kv_indptr"], is_causal=True)
    if kind == "step":
        s["graph"].replay()
        return {"logits": s["logits"], **_held(s["cache"])}
    s["cache"].reset()
    with torch.no_grad(), w8a8.int8_autocast(case["model"] == "dense"):
        logits = s["model"](s["ids"], s["cache"], logits_at=s["last"])["logits"]
    return {"logits": logits, **_held(s["cache"])}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def _layer_matrices(name):
    """Weight elements of the matrix products of a forward, layer runs counted as often as they run, and the head."""
    d, ff = WIDTH, 3 * WIDTH * FF
    if name == "dense":
        return LAYERS * (d * d * 2 + d * d // 2 + ff)
    if name == "lugitar":
        q, latent, kv = d * 16 * 192, d * 576, 16 * 256 * 512
        return 2 * (q + kv + d * d) + latent + 2 * 5 * d * d + 4 * ff
    rglru, delta = 3 * d * d + 2 * d * 256, 4 * d * d + 4 * d * 128
    return 3 * rglru + 2 * delta + (3 * d * d + d * d // 2) + 6 * ff + 3 * d * d


def work(case):
    kind = case["kind"]
    if kind in ("linear_int8", "linear_fp8", "linear_block"):
        m, k, n = case["tokens"], case["k"], case["n"]
        return {"bytes": 2 * m * k + n * k + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "train_fp8":
        m, k, n = case["tokens"], case["k"], case["n"]
        return {"bytes": 4 * (m * k + n * k + m * n), "flops": 6 * m * n * k}
    if kind in ("prompt_attn", "decode_attn"):
        h, g, d = case["heads"], case["kv_heads"], case["dim"]
        if kind == "decode_attn":
            new = [1] * case["batch"]
            kv = [max(1, int(case["context"] * s)) for s in _lengths(case)]
        elif case["paged"]:
            share = _lengths(case)
            new = [max(1, int(case["new"] * s)) for s in share]
            kv = [n + int(case["cached"] * s) for n, s in zip(new, reversed(share))]
        else:
            new = kv = [case["new"]] * case["batch"]
        seen = sum(n * m - n * (n - 1) // 2 for n, m in zip(new, kv))
        return {"bytes": 4 * sum(new) * h * d + 4 * sum(kv) * g * d, "flops": 4 * h * d * seen}
    batch, seq, name = case["batch"], case["seq"], case["model"]
    new = 1 if kind == "step" else seq
    matrices, head = _layer_matrices(name), WIDTH * VOCAB
    seen = (seq + 1) if new == 1 else seq * (seq + 1) // 2
    # per token in the dense decoder: scores and values of its layers; latent attention in two, a window of 1024
    # keys; one layer of attention beside 128 x 128 states per head elsewhere
    if name == "dense":
        mix, held = LAYERS * 4 * WIDTH * seen, LAYERS * 2 * 2 * (WIDTH // 4)
    elif name == "lugitar":
        near = min(seq + 1, 1024) if new == 1 else sum(min(i + 1, 1024) for i in range(seq))
        mix, held = 2 * 2 * 16 * 320 * near + 2 * new * 4 * 16 * 128 * 128, 2 * 576
    else:
        mix, held = 4 * WIDTH * seen + 2 * new * 6 * 16 * 128 * 128, 2 * 2 * (WIDTH // 4)
    stored = (matrices + head) * (1 if name == "dense" else 2)
    if name == "sarulix":   # weights of the layers that run twice are read once
        stored -= 2 * (3 * WIDTH * WIDTH + 2 * WIDTH * 256 + 4 * WIDTH * WIDTH + 4 * WIDTH * 128 + 6 * WIDTH * FF + WIDTH * WIDTH)
    return {"bytes": stored + batch * held * (seq + 1 if new == 1 else seq) + 2 * batch * VOCAB,
            "flops": batch * (2 * new * matrices + 2 * head + mix)}


def tolerance(case):
    # measured against `exact`; bf16 outputs of fp32 sums are 1.7e-3 off, a model's logits after its layers' roundings
    # (and, in int8, re-rounded codes) several times that
    return {"linear_int8": {"rel": 7e-3, "max": 0.06}, "linear_fp8": {"rel": 7e-3, "max": 0.06},
            "train_fp8": {"rel": 7e-3, "max": 0.06}, "linear_block": {"rel": 7e-3, "max": 0.06},
            "prompt_attn": {"rel": 1e-2, "max": 0.1}, "decode_attn": {"rel": 1e-2, "max": 0.1},
            "prompt": {"rel": 0.03, "max": 0.99}, "step": {"rel": 0.03, "max": 0.99}}[case["kind"]]


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------

def _divided(peak, most):
    """The fp32 quotient, rounded once."""
    return (peak.double().clamp_min(1e-12) / most).float()


def _int8_rows(x):
    """Codes of a symmetric per-row quantizer and its steps (which are defined in fp32)."""
    step = _divided(x.abs().amax(-1, keepdim=True), 127).double()
    return (x / step).round().clamp(-127, 127), step


def _int8_product(x, w):
    (a, sa), (b, sb) = _int8_rows(x), _int8_rows(w)
    return a @ b.t() * sa * sb.t()


def _fp8_codes(x, step, fmt):
    dtype, most = (torch.float8_e4m3fn, 448.0) if fmt == "e4m3" else (torch.float8_e5m2, 57344.0)
    return (x.detach().float() / step).clamp(-most, most).to(dtype).double()


def _step_of(x, most, seeded=False):
    """The quantization step of a tensor. ``seeded``: as the first call under delayed scaling forms it, dividing a
    tensor by a number (torch multiplies by the rounded reciprocal)."""
    peak = x.detach().abs().amax().float().clamp_min(1e-12)
    return peak / most if seeded else _divided(peak, most)


def _exact_linear(case, seed):
    x, w, b, g = _linear_inputs(case, seed)
    if case["kind"] == "linear_int8":
        out = _int8_product(x.double(), w.double())
        return out if b is None else out + b.double()
    if case["kind"] == "linear_block":
        m, k = x.shape
        n = w.size(0)
        out = torch.zeros(m, n, dtype=torch.float64, device=DEV)
        pad = F.pad(w, (0, 0, 0, -n % 128))
        for at in range(0, k, 128):
            part, rows = x[:, at:at + 128], pad[:, at:at + 128].reshape(-1, 128, 128)
            sx, sw = _divided(part.abs().amax(1, keepdim=True), 448), _divided(rows.abs().amax((1, 2), keepdim=True), 448)
            cx, cw = _fp8_codes(part, sx, "e4m3"), _fp8_codes(rows, sw, "e4m3") * sw.double()
            out += (cx * sx.double()) @ cw.reshape(-1, 128)[:n].t()
        return out
    delayed = not case["dynamic"]
    sx, sw = _step_of(x, 448.0, delayed), _step_of(w, 448.0, delayed)
    x8, w8 = _fp8_codes(x, sx, "e4m3"), _fp8_codes(w, sw, "e4m3")
    out = x8 @ w8.t() * (sx.double() * sw.double())
    if b is not None:
        out += b.double()
    if case["kind"] == "linear_fp8":
        return out
    if case["n"] != case["k"]:   # the fp8 backward takes square weights; others keep the bf16 products
        grads = [g.double() @ w.double(), g.double().t() @ x.double()]
        return {"out": out, "grads": tuple(grads + ([g.double().sum(0)] if b is not None else []))}
    # gradients in e5m2: delayed scaling keeps the steps that the forward recorded, dynamic scaling measures anew
    most = 448.0 if delayed else 57344.0
    sx, sw, sg = _step_of(x, most), _step_of(w, most), _step_of(g, 57344.0, delayed)
    x8, w8, g8 = (_fp8_codes(t, s, "e5m2") for t, s in ((x, sx), (w, sw), (g, sg)))
    grads = [g8 @ w8 * (sg.double() * sw.double()), g8.t() @ x8 * (sg.double() * sx.double())]
    return {"out": out, "grads": tuple(grads + ([g.double().sum(0)] if b is not None else []))}


def _attend(q, k, v, scale, seen, cap=None, sink=False):
    """``q [n, heads, d]``, ``k``, ``v [m, groups, d]``; ``seen [n, m]``, True where a query sees a key."""
    rep = q.size(1) // k.size(1)
    out = torch.empty(q.size(0), q.size(1), v.size(-1), dtype=torch.float64, device=q.device)
    for h in range(q.size(1)):
        s = q[:, h] @ k[:, h // rep].t() * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(~seen, float("-inf"))
        if sink:
            top = s.amax(-1, keepdim=True).clamp_min(0)
            e = torch.exp(s - top)
            p = e / (e.sum(-1, keepdim=True) + torch.exp(-top))
        else:
            p = torch.softmax(s, -1)
        out[:, h] = p @ v[:, h // rep]
    return out


def _causal(n, m, window=None):
    back = torch.arange(m - n, m, device=DEV)[:, None] - torch.arange(m, device=DEV)[None, :]
    return (back >= 0) if window is None else (back >= 0) & (back < window)


def _exact_attention(case, seed):
    scale = case["dim"] ** -0.5
    if case["kind"] == "prompt_attn" and not case["paged"]:
        s = _prompt_attn_inputs(case, seed)
        seen = _causal(case["new"], case["new"])
        return torch.stack([_attend(*(s[t][i].double() for t in "qkv"), scale, seen) for i in range(case["batch"])])
    if case["kind"] == "decode_attn":
        s = _decode_attn_inputs(case, seed)
        new = [1] * case["batch"]
    else:
        s = _prompt_attn_inputs(case, seed)
        new = s["new"]
    out, at = [], 0
    for i, (n, m) in enumerate(zip(new, s["kv"])):
        slots = s["table"][i, :m].long()
        out.append(_attend(s["q"][at:at + n].double(), s["k"][slots].double(), s["v"][slots].double(), scale, _causal(n, m)))
        at += n
    return torch.cat(out)


def _rotary(x, dims, base, adjacent=False, scaling=None):
    """``x [batch, tokens, heads, d]``: pairs of the first ``dims`` entries turned by position times frequency."""
    f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=x.device) / dims)
    size = 1.0
    if scaling is not None:
        def pair(turns):
            return dims * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
        lo, hi = max(math.floor(pair(scaling["fast"])), 0), min(math.ceil(pair(scaling["slow"])), dims - 1)
        keep = 1 - ((torch.arange(dims // 2, device=x.device).double() - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f = f * keep + f / scaling["factor"] * (1 - keep)
        size = 0.1 * math.log(scaling["factor"]) + 1.0
    angle = torch.outer(torch.arange(x.size(1), dtype=torch.float64, device=x.device), f)[:, None, :]
    cos, sin = torch.cos(angle) * size, torch.sin(angle) * size
    if adjacent:
        a, b = x[..., 0:dims:2], x[..., 1:dims:2]
        return torch.cat([torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2), x[..., dims:]], -1)
    a, b = x[..., :dims // 2], x[..., dims // 2:dims]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., dims:]], -1)


def _rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, eps):
    d = x - x.mean(-1, keepdim=True)
    return _rms(d, eps) * w


def _each(q, k, v, *rest, **more):
    return torch.stack([_attend(q[i], k[i], v[i], *rest, **more) for i in range(q.size(0))])


def _exact_dense(w, ids):
    (b, n), d, heads = ids.shape, WIDTH, HEAD_COUNT
    seen = _causal(n, n)

    def linear(x, *names):
        return _int8_product(x.reshape(b * n if x.size(1) == n else b, -1), torch.cat([w[t + ".weight"] for t in names]))

    x = w["embed_tokens.weight"][ids]
    for i in range(LAYERS):
        p = f"layers.{i}."
        h = _rms(x, 1e-5) * w[p + "input_norm.weight"]
        q, k, v = linear(h, *(p + f"attention.{t}_proj" for t in "qkv")).reshape(b, n, -1, d // heads).split(
            [heads, heads // 4, heads // 4], 2)
        q, k = (_rotary(t, d // heads, 10000.0, adjacent=True) for t in (q, k))
        o = _each(q, k, v, (d // heads) ** -0.5, seen).reshape(b, n, d)
        x = x + linear(o, p + "attention.o_proj").reshape(b, n, d)
        gate, up = linear(_rms(x, 1e-5) * w[p + "post_attention_norm.weight"], p + "mlp.gate", p + "mlp.up").chunk(2, -1)
        x = x + linear((F.silu(gate) * up).reshape(b, n, -1), p + "mlp.down").reshape(b, n, d)
    x = _rms(x[:, -1:], 1e-5) * w["norm.weight"]
    return _int8_product(x.reshape(b, d), w["lm_head.weight"]).reshape(b, 1, -1), []


def _exact_lugitar(w, ids, cfg):
    (b, n), eps = ids.shape, cfg["norm"]["eps"]
    x, states, latents = w["embed"][ids], [], None
    for i, layer in enumerate(cfg["layers"]):
        p, m = f"l{i}.mix.", layer["mixer"]
        heads, d, vd = m["heads"], m["dim"], m["vdim"]
        h = _layer_norm(x, w[f"l{i}.norm1"], eps)
        if layer["type"] == "latent_attention":
            rot = m["rot"]
            turn = lambda t: _rotary(t, rot["dims"], rot["base"], scaling=rot["scaling"])  # noqa: E731
            if "kv_from" not in m:
                c, r = (h @ w[p + "dkv"].t()).split([m["kv_rank"], m["rot_dim"]], -1)
                latents = _rms(c, eps) * w[p + "dkv.norm"], turn(r[:, :, None])
            c, r = latents
            q, qr = (h @ w[p + "q"].t()).reshape(b, n, heads, -1).split([d, m["rot_dim"]], -1)
            q = torch.cat([q, turn(qr)], -1)
            k = torch.cat([(c @ w[p + "uk"].t()).reshape(b, n, heads, d), r.expand(b, n, heads, -1)], -1)
            v = (c @ w[p + "uv"].t()).reshape(b, n, heads, vd)
            o = _each(q, k, v, m["scale"], _causal(n, n, m["mask"]["size"]))
            o = (o * torch.sigmoid(h @ w[p + "g"].t())[..., None]).reshape(b, n, -1)
        else:
            q, k, v = (F.silu(h @ w[p + t].t()).reshape(b, n, heads, -1) for t in "qkv")
            s = torch.zeros(b, heads, d, vd, dtype=torch.float64, device=DEV)
            lam = torch.tensor(m["decay"], dtype=torch.float64, device=DEV).reshape(1, heads, 1, 1)
            o = torch.empty(b, n, heads, vd, dtype=torch.float64, device=DEV)
            for t in range(n):
                s = torch.addcmul(s * lam, k[:, t, :, :, None], v[:, t, :, None, :])
                o[:, t] = (s * q[:, t, :, :, None]).sum(2)
            states.append(s)
            o = _rms(o.reshape(b, n, -1), eps) * w[p + "norm"] * torch.sigmoid(h @ w[p + "g"].t())
        x = x + cfg["residual_mult"] * _layer_norm(o @ w[p + "o"].t(), w[f"l{i}.norm1b"], eps)
        h = _layer_norm(x, w[f"l{i}.norm2"], eps)
        y = (F.silu(h @ w[f"l{i}.mlp.gate"].t()) * (h @ w[f"l{i}.mlp.up"].t())) @ w[f"l{i}.mlp.down"].t()
        x = x + cfg["residual_mult"] * _layer_norm(y, w[f"l{i}.norm2b"], eps)
    return _layer_norm(x[:, -1:], w["final.norm"], eps) @ w["head"].t(), states


def _short_conv(x, taps):
    n, t = x.size(1), taps.size(1)
    padded = F.pad(x, (0, 0, t - 1, 0))
    return sum(padded[:, j:j + n] * taps[:, j] for j in range(t))


def _unit(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _sarulix_mixer(kind, h, w, p, m, eps):
    b, n, _ = h.shape
    if kind == "attention":
        heads, groups, d, rot = m["heads"], m["kv_heads"], m["dim"], m["rot"]
        q, k, v = ((h @ w[p + t].t() + w[p + t + ".b"]).reshape(b, n, c, -1) for t, c in (("q", heads), ("k", groups), ("v", groups)))
        q, k = (_rotary(_rms(t, eps) * w[p + c + ".norm"], rot["dims"], rot["base"]) for t, c in ((q, "q"), (k, "k")))
        o = _each(q, k, v, m["scale"], _causal(n, n), cap=m["softcap"], sink=True).reshape(b, n, -1)
        return (o * torch.sigmoid(h @ w[p + "g"].t())) @ w[p + "o"].t() + w[p + "o.b"], None
    if kind == "rglru":
        y = F.gelu(h @ w[p + "y"].t() + w[p + "y.b"], approximate="tanh")
        u = _short_conv(h @ w[p + "x"].t() + w[p + "x.b"], w[p + "conv"]) + w[p + "conv.b"]
        part = u.reshape(b * n, m["blocks"], -1)
        r, i = (torch.sigmoid(torch.stack([part[:, j] @ w[p + t][j].t() for j in range(m["blocks"])], 1) + w[p + t + ".b"])
                .reshape(b, n, -1) for t in ("ra", "ri"))
        log_a = -8 * r * F.softplus(w[p + "lam"])
        a, fresh = torch.exp(log_a), torch.sqrt(-torch.expm1(2 * log_a)) * i * u
        s, o = torch.zeros_like(u[:, 0]), torch.empty_like(u)
        for t in range(n):
            s = torch.addcmul(fresh[:, t], a[:, t], s)
            o[:, t] = s
        return (o * y) @ w[p + "o"].t(), s
    heads, d = m["heads"], m["dim"]
    q, k, v = (F.silu(_short_conv(h @ w[p + t].t(), w[p + t + ".conv"])).reshape(b, n, heads, -1) for t in "qkv")
    q, k = _unit(q) * d ** -0.5, _unit(k)
    beta = torch.sigmoid(h @ w[p + "b"].t())
    dt = F.softplus(h @ w[p + "a1"].t() @ w[p + "a2"].t() + w[p + "dt_bias"]).reshape(b, n, heads, d)
    g = torch.exp(-torch.exp(w[p + "A_log"])[:, None] * dt)
    s = torch.zeros(b, heads, d, m["vdim"], dtype=torch.float64, device=DEV)
    o = torch.empty_like(v)
    for t in range(n):
        s = s * g[:, t, :, :, None]
        u = beta[:, t, :, None] * (v[:, t] - (s * k[:, t, :, :, None]).sum(2))
        s = torch.addcmul(s, k[:, t, :, :, None], u[:, :, None, :])
        o[:, t] = (s * q[:, t, :, :, None]).sum(2)
    gate = torch.sigmoid(h @ w[p + "g1"].t() @ w[p + "g2"].t()).reshape(b, n, heads, -1)
    return (_rms(o, eps) * w[p + "norm"] * gate).reshape(b, n, -1) @ w[p + "o"].t(), s


def _exact_sarulix(w, ids, cfg):
    eps, loop = cfg["norm"]["eps"], cfg["loop"]
    x = x0 = w["embed"][ids]
    order = [(i, None) for i in range(loop["start"])]
    order += [(i, t if i == loop["start"] else None) for t in range(loop["times"]) for i in range(loop["start"], loop["stop"])]
    order += [(i, None) for i in range(loop["stop"], len(cfg["layers"]))]
    states = []
    for i, opens in order:
        layer = cfg["layers"][i]
        if opens is not None:
            x = torch.cat([x, x0], -1) @ w["loop.in"].t() + w["loop.step"][opens]
        y, s = _sarulix_mixer(layer["type"], _rms(x, eps) * (1 + w[f"l{i}.norm1"]), w, f"l{i}.mix.", layer["mixer"], eps)
        states += [] if s is None else [s]
        x = x + y
        h = _rms(x, eps) * (1 + w[f"l{i}.norm2"])
        x = x + (F.gelu(h @ w[f"l{i}.mlp.gate"].t(), approximate="tanh") * (h @ w[f"l{i}.mlp.up"].t())) @ w[f"l{i}.mlp.down"].t()
    return _rms(x[:, -1:], eps) * (1 + w["final.norm"]) @ w["head"].t() * cfg["logit_scale"], states


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear_int8", "linear_fp8", "train_fp8", "linear_block"):
        return _exact_linear(case, seed)
    if kind in ("prompt_attn", "decode_attn"):
        return _exact_attention(case, seed)
    w = {name: t.double() for name, t in _weights(case["model"], seed).items()}
    ids = _prompt_ids(case, seed, 1)
    ids = ids if kind == "step" else ids[:, :-1]
    if case["model"] == "dense":
        logits, states = _exact_dense(w, ids)
        return {"logits": logits, "rows": [None, None]}
    logits, states = (_exact_lugitar if case["model"] == "lugitar" else _exact_sarulix)(w, ids, _config(case["model"]))
    return {"logits": logits, "state": states, "rows": None}
