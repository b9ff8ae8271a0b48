"""The work a user of simple_llm_amd has it do, as a list of measurable cases.

Every case goes through the package's public entry points, as a serving or
training program calls them:

  decode    one or more decode steps of an attention layer over its KV cache:
            kv_cache_append_attend, or the reference's pair kv_cache_update +
            attention_with_kv_cache
  prefill   a chunk of prompt tokens into a layer's cache with its causal
            attention: kv_cache_prefill
  train     flash_attention and flash_attention_backward of a layer
  forward   the logits of every position of a batch: backend.forward
  step      decode steps of the whole model on given tokens:
            TransformerModel.forward_step
  generate  a whole greedy generation, prompts to tokens: Generator.run
  sample    one token from a logits row: backend.sample_token

Sizes are those of the repository's benchmark workloads (bench.py) and of the
model shapes its tests use; draw() spreads them over the ranges between.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "llm-experiments_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda:0"
_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}
_BYTES = {"fp32": 4, "bf16": 2}


def listed():
    return [
        # Long-context serving: 4 sequences at 32K filled positions, bf16 cache.
        # The cache read is everything; the repository's headline workload.
        {"name": "decode_long", "kind": "decode", "batch": 4, "kv_heads": 16, "groups": 1,
         "head_dim": 128, "dtype": "bf16", "fill": 32000, "lens": "equal", "page": 0,
         "api": "fused", "steps": 4},
        # A small fp32 cache with sequences of every length (the reference's
        # default storage): 20 us calls, where launches and host work count.
        {"name": "decode_small", "kind": "decode", "batch": 8, "kv_heads": 8, "groups": 1,
         "head_dim": 64, "dtype": "fp32", "fill": 2040, "lens": "uniform", "page": 0,
         "api": "fused", "steps": 8},
        # Batched serving of a grouped-query model from a paged cache, ragged
        # lognormal lengths.
        {"name": "decode_paged_gqa", "kind": "decode", "batch": 64, "kv_heads": 8, "groups": 4,
         "head_dim": 128, "dtype": "bf16", "fill": 8192, "lens": "lognormal", "page": 16,
         "api": "fused", "steps": 4},
        # A 512-token chunk of four long prompts, onto a 32K prefix.
        {"name": "prefill_long", "kind": "prefill", "batch": 4, "kv_heads": 16, "groups": 1,
         "head_dim": 128, "dtype": "bf16", "prefix": 32256, "chunk": 512, "ragged": False},
        # Short ragged prompts of a grouped-query model, as a server admits
        # them: chunk lengths and prefixes differ by sequence.
        {"name": "prefill_ragged_gqa", "kind": "prefill", "batch": 6, "kv_heads": 8, "groups": 4,
         "head_dim": 128, "dtype": "bf16", "prefix": 1900, "chunk": 333, "ragged": True},
        # Training attention, forward and backward, at the repository's
        # training shape.
        {"name": "train_attention", "kind": "train", "batch": 8, "seq": 2048, "heads": 16,
         "head_dim": 64},
        # The same for a small model (d 384, 8 heads) on an odd context.
        {"name": "train_attention_small", "kind": "train", "batch": 4, "seq": 333, "heads": 8,
         "head_dim": 48},
        # Scoring: logits of every position of two full windows, GPT-2-small
        # shape.
        {"name": "forward_gpt2", "kind": "forward", "layers": 12, "heads": 12, "head_dim": 64,
         "vocab": 50304, "context": 1024, "batch": 2, "tokens": 1024},
        # Decode steps of that model on given tokens (constrained decoding),
        # batch 16, bf16 cache.
        {"name": "step_gpt2", "kind": "step", "layers": 12, "heads": 12, "head_dim": 64,
         "vocab": 50304, "context": 1024, "batch": 16, "fill": 700, "dtype": "bf16",
         "steps": 4},
        # Generation with that model: 16 ragged prompts prefilled together,
        # then the captured decode step replayed.
        {"name": "generate_gpt2", "kind": "generate", "layers": 12, "heads": 12, "head_dim": 64,
         "vocab": 50304, "context": 1024, "batch": 16, "prompt": 512, "new": 32},
        # Generation with a byte-level tiny model, batch 1: short kernels, so
        # their number decides.
        {"name": "generate_tiny", "kind": "generate", "layers": 4, "heads": 4, "head_dim": 64,
         "vocab": 256, "context": 256, "batch": 1, "prompt": 64, "new": 192},
        # One filtered draw from a GPT-2 vocabulary row, the smallest call.
        {"name": "sample_filtered", "kind": "sample", "vocab": 50304, "temperature": 0.8,
         "top_k": 40, "top_p": 0.95, "min_p": 0.02, "penalty": 1.1, "recent": 64},
    ]


# ---------------------------------------------------------------------------
# Drawn cases
# ---------------------------------------------------------------------------

_HEAD_DIMS = [24, 32, 48, 64, 64, 64, 80, 96, 128, 128, 128]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 3 + ["train"] * 3 + ["forward"] * 2
                      + ["step", "generate", "sample"])
    while True:
        case = _DRAW[kind](rng)
        w = work(case)
        most = _MOST[kind]
        if kind == "prefill" and case["dtype"] == "fp32":
            most = (most[0], 5e10)
        if w["bytes"] <= most[0] and w["flops"] <= most[1]:
            return case


#: The most bytes and flops of a drawn case, by kind (the largest listed ones').
_MOST = {"decode": (4.2e9, 1e12), "prefill": (1.3e9, 5e11), "train": (1e9, 2.4e11),
         "forward": (2e9, 6e11), "step": (3e9, 1e11), "generate": (5e10, 1e12),
         "sample": (1e9, 1e9)}


def _draw_decode(rng):
    hkv = rng.choice([1, 2, 4, 8, 8, 12, 16])
    g = rng.choice([1, 1, 2, 4, 8])
    return {"kind": "decode", "batch": _log(rng, 1, 64), "kv_heads": hkv, "groups": g,
            "head_dim": rng.choice(_HEAD_DIMS), "dtype": rng.choice(["fp32", "bf16", "bf16"]),
            "fill": _log(rng, 64, 32768), "lens": rng.choice(["equal", "uniform", "lognormal"]),
            "page": rng.choice([0, 0, 16]), "api": rng.choice(["fused", "fused", "pair"]),
            "steps": 4}


def _draw_prefill(rng):
    dtype = rng.choice(["fp32", "bf16", "bf16"])
    # (a bf16 cache at head_dim 32 had no prefill kernel when these ranges were set)
    dims = [d for d in _HEAD_DIMS if dtype == "fp32" or d != 32]
    return {"kind": "prefill", "batch": _log(rng, 1, 8),
            "kv_heads": rng.choice([2, 4, 8, 12, 16]), "groups": rng.choice([1, 1, 2, 4, 8]),
            "head_dim": rng.choice(dims), "dtype": dtype,
            "prefix": rng.choice([0, _log(rng, 16, 32000)]), "chunk": _log(rng, 17, 1024),
            "ragged": rng.choice([True, False])}


def _draw_train(rng):
    return {"kind": "train", "batch": _log(rng, 1, 16), "seq": _log(rng, 33, 2048),
            "heads": rng.choice([2, 4, 6, 8, 12, 16]), "head_dim": rng.choice(_HEAD_DIMS)}


def _draw_model(rng):
    return {"layers": rng.choice([2, 4, 6, 8, 12]), "heads": rng.choice([2, 4, 6, 8, 12]),
            "head_dim": rng.choice([24, 32, 48, 64, 64, 80]), "vocab": _log(rng, 256, 50304)}


def _draw_forward(rng):
    t = _log(rng, 48, 1024)
    return {"kind": "forward", **_draw_model(rng), "context": t + rng.choice([0, 0, 64]),
            "batch": _log(rng, 1, 8), "tokens": t}


def _draw_step(rng):
    fill = _log(rng, 16, 1000)
    return {"kind": "step", **_draw_model(rng), "context": 1024, "batch": _log(rng, 1, 16),
            "fill": fill, "dtype": rng.choice(["fp32", "bf16"]), "steps": 4}


def _draw_generate(rng):
    return {"kind": "generate", **_draw_model(rng), "context": 1024, "batch": _log(rng, 1, 16),
            "prompt": _log(rng, 8, 512), "new": _log(rng, 8, 64)}


def _draw_sample(rng):
    return {"kind": "sample", "vocab": _log(rng, 256, 65536),
            "temperature": round(rng.uniform(0.5, 1.3), 2),
            "top_k": rng.choice([0, _log(rng, 4, 200)]), "top_p": rng.choice([1.0, 0.9, 0.95]),
            "min_p": rng.choice([0.0, 0.02]), "penalty": rng.choice([1.0, 1.1]),
            "recent": rng.choice([0, 64])}


_DRAW = {"decode": _draw_decode, "prefill": _draw_prefill, "train": _draw_train,
         "forward": _draw_forward, "step": _draw_step, "generate": _draw_generate,
         "sample": _draw_sample}


# ---------------------------------------------------------------------------
# Inputs, from the seed alone
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _lengths(kind, n, top, seed):
    """n sequence lengths in [1, top]; the longest is top, as a batch is
    admitted against its limit."""
    r = np.random.default_rng(int(seed))
    if kind == "equal":
        lens = np.full(n, top)
    elif kind == "uniform":
        lens = r.integers(1, top + 1, n)
    else:  # lognormal around 1500 of 8192, in proportion
        lens = np.clip(np.exp(r.normal(math.log(max(top * 1500 / 8192, 1)), 0.8, n)),
                       min(16, top), top)
    lens = lens.astype(np.int64)
    lens[int(r.integers(n))] = top
    return lens


def _cache_rows(g, rows, width, dtype):
    out = torch.empty((rows, width), dtype=dtype, device=DEV)
    for i in range(0, rows, 1 << 16):
        part = out[i:i + (1 << 16)]
        part.copy_(torch.randn(part.shape, generator=g, device=DEV))
    return out


def _decode_inputs(c, seed):
    g = _gen(seed)
    hkv, hq, d = c["kv_heads"], c["kv_heads"] * c["groups"], c["head_dim"]
    lens = _lengths(c["lens"], c["batch"], c["fill"], seed)
    cap = c["fill"] + c["steps"]
    table = None
    if c["page"]:
        per = -(-cap // c["page"])
        pages = c["batch"] * per
        perm = np.random.default_rng(int(seed) + 1).permutation(pages)
        table = perm.reshape(c["batch"], per).astype(np.int32)
        rows = pages * c["page"]
    else:
        rows = c["batch"] * cap
    dt = _DTYPES[c["dtype"]]
    return {"k": _cache_rows(g, rows, hkv * d, dt), "v": _cache_rows(g, rows, hkv * d, dt),
            "lens": lens, "cap": cap, "table": table,
            "q": _randn(g, c["steps"], c["batch"], hq, d),
            "nk": _randn(g, c["steps"], c["batch"], hkv, d),
            "nv": _randn(g, c["steps"], c["batch"], hkv, d)}


def _prefill_inputs(c, seed):
    g = _gen(seed)
    hkv, hq, d, n, ch = (c["kv_heads"], c["kv_heads"] * c["groups"], c["head_dim"], c["batch"],
                         c["chunk"])
    start = np.full(n, c["prefix"], np.int64)
    count = np.full(n, ch, np.int64)
    if c["ragged"]:
        if c["prefix"]:
            start = _lengths("uniform", n, c["prefix"], seed)
        count = _lengths("uniform", n, ch, seed + 1)
    cap = c["prefix"] + ch
    dt = _DTYPES[c["dtype"]]
    return {"k": _cache_rows(g, n * cap, hkv * d, dt), "v": _cache_rows(g, n * cap, hkv * d, dt),
            "start": start, "count": count, "cap": cap, "q": _randn(g, n, ch, hq, d),
            "nk": _randn(g, n, ch, hkv, d), "nv": _randn(g, n, ch, hkv, d)}


def _train_inputs(c, seed):
    g = _gen(seed)
    shape = (c["batch"] * c["seq"], c["heads"] * c["head_dim"])
    return [_randn(g, *shape) for _ in range(4)]  # q, k, v, grad of the output


def _position_table(n, d):
    pos = np.arange(n, dtype=np.float64)[:, None]
    i = np.arange(d)[None, :]
    ang = pos / (10000.0 ** (2 * (i // 2) / d))
    return np.concatenate([np.sin(ang[:, 0::2]), np.cos(ang[:, 1::2])], -1).astype(np.float32)


def _weights(c, seed):
    """N(0, 0.02) matrices, LayerNorm gains around 1, small biases (device
    tensors, the reference's field names and [in, out] layout)."""
    g = _gen(seed)
    d = c["heads"] * c["head_dim"]

    def w(*shape, std=0.02, mean=0.0):
        return _randn(g, *shape) * std + mean

    layers = []
    for _ in range(c["layers"]):
        layers.append({
            "attn_wq": w(d, d), "attn_wk": w(d, d), "attn_wv": w(d, d), "attn_wo": w(d, d),
            "ff_w1": w(d, 4 * d), "ff_b1": w(4 * d), "ff_w2": w(4 * d, d), "ff_b2": w(d),
            "ln_gamma1": w(d, std=0.1, mean=1.0), "ln_beta1": w(d),
            "ln_gamma2": w(d, std=0.1, mean=1.0), "ln_beta2": w(d)})
    return {"embedding": w(c["vocab"], d),
            "pos_encoding": torch.from_numpy(_position_table(c["context"], d)).to(DEV),
            "layers": layers}


def _on_host(p):
    out = {k: p[k].cpu().numpy() for k in ("embedding", "pos_encoding")}
    out["layers"] = [{k: t.cpu().numpy() for k, t in lp.items()} for lp in p["layers"]]
    return out


def _tokens(c, seed, *shape):
    return np.random.default_rng(int(seed) + 3).integers(0, c["vocab"], shape)


def _prompts(c, seed):
    lens = _lengths("uniform", c["batch"], c["prompt"], c["prompt"])  # the case's own
    lens = np.maximum(lens, min(32, c["prompt"]))
    ids = _tokens(c, seed, c["batch"], c["prompt"])
    return [ids[b, :n].tolist() for b, n in enumerate(lens)]


def _sample_inputs(c, seed):
    logits = _randn(_gen(seed), c["vocab"]) * 2.5  # a language model's spread
    recent = _tokens(c, seed, c["recent"])
    return logits, recent


# ---------------------------------------------------------------------------
# prepare: what a program has in hand before the call
# ---------------------------------------------------------------------------

def prepare(case, seed):
    return _PREPARE[case["kind"]](dict(case), int(seed))


def _prepare_decode(c, seed):
    from simple_llm_amd.gpu import gpu

    ctx = gpu.context_create()
    x = _decode_inputs(c, seed)
    hkv, hq, d = c["kv_heads"], c["kv_heads"] * c["groups"], c["head_dim"]
    cache = gpu.kv_cache_create(ctx, gpu.KVCacheConfig(
        c["batch"], x["cap"], 1, hq, d, n_kv_heads=hkv, dtype=_DTYPES[c["dtype"]],
        block_size=c["page"], n_blocks=x["k"].shape[0] // c["page"] if c["page"] else 0))
    if c["page"]:
        gpu.kv_cache_set_block_table(cache, torch.from_numpy(x["table"]))
    layer = cache.layers[0]
    layer.k_cache.buffer.copy_(x["k"])
    layer.v_cache.buffer.copy_(x["v"])
    s = {"case": c, "gpu": gpu, "ctx": ctx, "cache": cache, "host": x["lens"],
         "lens": torch.from_numpy(x["lens"].astype(np.int32)).to(DEV)}
    out = [torch.empty_like(x["q"][0]) for _ in range(c["steps"])]
    if c["api"] == "pair":
        def flat(t):
            return gpu.gpu_buffer_from_tensor(t.reshape(c["batch"], -1))
        s["steps"] = [tuple(flat(t) for t in (x["nk"][i], x["nv"][i], x["q"][i], out[i]))
                      for i in range(c["steps"])]
    else:
        s["steps"] = [(x["nk"][i], x["nv"][i], x["q"][i], out[i]) for i in range(c["steps"])]
    s["out"] = out
    return s


def _prepare_prefill(c, seed):
    from simple_llm_amd.gpu import gpu

    ctx = gpu.context_create()
    x = _prefill_inputs(c, seed)
    cache = gpu.kv_cache_create(ctx, gpu.KVCacheConfig(
        c["batch"], x["cap"], 1, c["kv_heads"] * c["groups"], c["head_dim"],
        n_kv_heads=c["kv_heads"], dtype=_DTYPES[c["dtype"]]))
    layer = cache.layers[0]
    layer.k_cache.buffer.copy_(x["k"])
    layer.v_cache.buffer.copy_(x["v"])
    return {"case": c, "gpu": gpu, "ctx": ctx, "cache": cache, "host": x["start"],
            "lens": torch.from_numpy(x["start"].astype(np.int32)).to(DEV), "nk": x["nk"],
            "nv": x["nv"], "q": x["q"], "out": torch.empty_like(x["q"]),
            "count": x["count"] if c["ragged"] else None}


def _prepare_train(c, seed):
    from simple_llm_amd.gpu import gpu

    ctx = gpu.context_create()
    rows, e = c["batch"] * c["seq"], c["heads"] * c["head_dim"]
    blocks = -(-c["seq"] // ctx.config.flash_attn_br)
    wrap = gpu.gpu_buffer_from_tensor

    def empty(*shape):
        return wrap(torch.empty(shape, device=DEV))

    q, k, v, go = (wrap(t) for t in _train_inputs(c, seed))
    return {"case": c, "gpu": gpu, "ctx": ctx, "q": q, "k": k, "v": v, "go": go,
            "o": empty(rows, e), "l": empty(rows * c["heads"]), "m": empty(rows * c["heads"]),
            "gq": empty(rows, e), "gk": empty(rows, e), "gv": empty(rows, e),
            "wk": empty(blocks * rows, e), "wv": empty(blocks * rows, e)}


def _model(c, seed, dtype="fp32"):
    from simple_llm_amd.gpu import gpu
    from simple_llm_amd.model import TransformerModel, TransformerModelParams

    tm = TransformerModelParams(c["vocab"], c["heads"] * c["head_dim"], c["context"], c["heads"],
                                c["layers"])
    return TransformerModel(gpu.context_create(), tm, _on_host(_weights(c, seed)),
                            kv_dtype=_DTYPES[dtype])


def _prepare_forward(c, seed):
    from simple_llm_amd import backend

    params = _on_host(_weights(c, seed))
    backend.device_model(params, c["layers"], c["heads"], c["head_dim"])
    return {"case": c, "backend": backend, "params": params,
            "tokens": _tokens(c, seed, c["batch"], c["tokens"])}


def _prepare_step(c, seed):
    model = _model(c, seed, c["dtype"])
    cache = model.new_cache(c["batch"])
    g = _gen(seed + 1)
    for layer in cache.layers:  # a cache of earlier tokens
        for buf in (layer.k_cache.buffer, layer.v_cache.buffer):
            buf.copy_(torch.randn(buf.shape, generator=g, device=DEV))
    ids = torch.from_numpy(_tokens(c, seed, c["steps"], c["batch"]).astype(np.int32)).to(DEV)
    return {"case": c, "model": model, "cache": cache, "ids": list(ids.unbind(0)),
            "out": torch.empty((c["steps"], c["batch"], c["vocab"]), device=DEV)}


def _prepare_generate(c, seed):
    from simple_llm_amd.model import Generator

    prompts = _prompts(c, seed)
    gen = Generator(_model(c, seed), prompts, [len(p) + c["new"] for p in prompts],
                    use_graph=True)
    return {"case": c, "gen": gen}


def _prepare_sample(c, seed):
    from simple_llm_amd import backend

    logits, recent = _sample_inputs(c, seed)
    return {"case": c, "backend": backend, "logits": logits, "recent": recent, "key": seed}


_PREPARE = {"decode": _prepare_decode, "prefill": _prepare_prefill, "train": _prepare_train,
            "forward": _prepare_forward, "step": _prepare_step, "generate": _prepare_generate,
            "sample": _prepare_sample}


# ---------------------------------------------------------------------------
# run: one pass
# ---------------------------------------------------------------------------

def run(state):
    return _RUN[state["case"]["kind"]](state)


def _rewind(s):
    """Back to the fills before the pass, as a server drops tokens it does
    not keep: one small copy."""
    layer = s["cache"].layers[0]
    layer.lens.copy_(s["lens"])
    layer.host_lens = s["host"].copy()


def _run_decode(s):
    _rewind(s)
    gpu, ctx, cache = s["gpu"], s["ctx"], s["cache"]
    if s["case"]["api"] == "pair":
        for k, v, q, out in s["steps"]:
            gpu.kv_cache_update(ctx, cache, 0, k, v)
            gpu.attention_with_kv_cache(ctx, cache, 0, q, out)
    else:
        for k, v, q, out in s["steps"]:
            gpu.kv_cache_append_attend(ctx, cache, 0, k, v, q, out)
    layer = cache.layers[0]
    return {"out": s["out"], "lens": layer.lens, "k": layer.k_cache.buffer,
            "v": layer.v_cache.buffer}


def _run_prefill(s):
    _rewind(s)
    cache = s["cache"]
    s["gpu"].kv_cache_prefill(s["ctx"], cache, 0, s["nk"], s["nv"], s["q"], s["out"],
                              n_new=s["count"])
    layer = cache.layers[0]
    return {"out": s["out"], "lens": layer.lens, "k": layer.k_cache.buffer,
            "v": layer.v_cache.buffer}


def _run_train(s):
    c, gpu, ctx = s["case"], s["gpu"], s["ctx"]
    dims = (c["batch"], c["seq"], c["heads"], c["head_dim"])
    gpu.flash_attention(ctx, s["q"], s["k"], s["v"], s["o"], s["l"], s["m"], *dims)
    gpu.flash_attention_backward(ctx, s["q"], s["k"], s["v"], s["o"], s["l"], s["m"], s["go"],
                                 s["gq"], s["wk"], s["wv"], s["gk"], s["gv"], *dims)
    return {n: s[n].buffer for n in ("o", "l", "m", "gq", "gk", "gv")}


def _run_forward(s):
    c = s["case"]
    return s["backend"].forward(s["params"], s["tokens"], c["layers"], c["heads"], c["head_dim"])


def _kv(cache):
    return [b.buffer for layer in cache.layers for b in (layer.k_cache, layer.v_cache)]


def _run_step(s):
    model, cache = s["model"], s["cache"]
    cache.current_len = s["case"]["fill"]
    for i, ids in enumerate(s["ids"]):
        s["out"][i].copy_(model.forward_step(cache, ids))
    return {"logits": s["out"], "lens": cache.layers[-1].lens, "kv": _kv(cache)}


def _run_generate(s):
    last = {}

    def keep(j, logits):
        last["logits"] = logits

    tokens = s["gen"].run(on_step=keep)
    return {"tokens": np.concatenate([np.asarray(t, np.int64) for t in tokens]),
            "logits": last["logits"], "kv": _kv(s["gen"].cache)}


def _run_sample(s):
    c = s["case"]
    return s["backend"].sample_token(s["key"], s["logits"], c["temperature"], c["top_k"],
                                     c["top_p"], c["min_p"], c["penalty"], s["recent"])


_RUN = {"decode": _run_decode, "prefill": _run_prefill, "train": _run_train,
        "forward": _run_forward, "step": _run_step, "generate": _run_generate,
        "sample": _run_sample}


# ---------------------------------------------------------------------------
# work: what the path cannot do without
# ---------------------------------------------------------------------------

def work(case):
    return _WORK[case["kind"]](case)


def _mean_fill(c):
    top = c["fill"]
    return {"equal": top, "uniform": top / 2, "lognormal": top * 0.25}[c["lens"]]


def _work_decode(c):
    d, hkv, hq, n = c["head_dim"], c["kv_heads"], c["kv_heads"] * c["groups"], c["steps"]
    total = c["batch"] * _mean_fill(c)
    rows = c["batch"] * d * (2 * hq * 4 + 2 * hkv * (4 + _BYTES[c["dtype"]]))
    return {"bytes": n * (2 * hkv * d * total * _BYTES[c["dtype"]] + rows),
            "flops": n * 4 * hq * d * total}


def _work_prefill(c):
    d, hkv, hq, s = c["head_dim"], c["kv_heads"], c["kv_heads"] * c["groups"], _BYTES[c["dtype"]]
    half = 0.5 if c["ragged"] else 1.0
    pre, new = c["prefix"] * half, c["chunk"] * half
    rows = c["batch"] * new
    return {"bytes": c["batch"] * 2 * hkv * d * pre * s + rows * d * (2 * hkv * (4 + s) + 8 * hq),
            "flops": 4 * d * hq * rows * (pre + new / 2)}


def _work_train(c):
    rows, e = c["batch"] * c["seq"], c["heads"] * c["head_dim"]
    pairs = c["batch"] * c["heads"] * c["seq"] * (c["seq"] + 1) / 2
    return {"bytes": 4 * rows * (8 * e + 2 * c["heads"]),
            "flops": 14 * c["head_dim"] * pairs}


def _matrix_params(c):
    d = c["heads"] * c["head_dim"]
    return c["layers"] * 12 * d * d, c["vocab"] * d


def _work_forward(c):
    body, head = _matrix_params(c)
    d, m = c["heads"] * c["head_dim"], c["batch"] * c["tokens"]
    return {"bytes": 4 * (body + head + m * c["vocab"]),
            "flops": 2 * m * (body + head)
            + 4 * d * c["layers"] * c["batch"] * c["tokens"] * (c["tokens"] + 1) / 2}


def _decode_step_work(c, fill, kv_bytes):
    body, head = _matrix_params(c)
    d = c["heads"] * c["head_dim"]
    kv = 2 * d * c["layers"] * c["batch"] * fill
    return (4 * (body + head + c["batch"] * c["vocab"]) + kv_bytes * kv,
            2 * c["batch"] * (body + head) + 2 * kv)


def _work_step(c):
    b, f = _decode_step_work(c, c["fill"], _BYTES[c["dtype"]])
    return {"bytes": c["steps"] * b, "flops": c["steps"] * f}


def _work_generate(c):
    body, head = _matrix_params(c)
    d, p = c["heads"] * c["head_dim"], c["prompt"] * (1.0 if c["batch"] == 1 else 0.5)
    b, f = _decode_step_work(c, p + c["new"] / 2, 4)
    rows = c["batch"] * p
    return {"bytes": 4 * (body + head) + (c["new"] - 1) * b,
            "flops": 2 * (rows * body + c["batch"] * head) + 2 * d * c["layers"] * rows * p
            + (c["new"] - 1) * f}


def _work_sample(c):
    return {"bytes": 4 * c["vocab"], "flops": 10 * c["vocab"]}


_WORK = {"decode": _work_decode, "prefill": _work_prefill, "train": _work_train,
         "forward": _work_forward, "step": _work_step, "generate": _work_generate,
         "sample": _work_sample}


# ---------------------------------------------------------------------------
# tolerance
# ---------------------------------------------------------------------------

def tolerance(case):
    k = case["kind"]
    if k == "sample":
        return "exact"
    if k == "prefill" and case["dtype"] == "bf16":
        # queries and probabilities enter the matrix core as bf16
        return {"rel": 1e-2, "max": 0.2}
    if k == "decode":
        # grouped queries enter the matrix core as two bf16 parts
        return {"rel": 2e-5, "max": 1e-3}
    if k == "generate":
        # a near tie may pick another token; its row's logits then differ
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.01}
    if k == "step" and case["dtype"] == "bf16":
        # a last-bit change of k or v moves its rounding into the bf16 cache
        return {"rel": 1e-4, "max": 1e-2}
    return {"rel": 1e-5, "max": 1e-3}


# ---------------------------------------------------------------------------
# exact: the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def exact(case, seed):
    return _EXACT[case["kind"]](dict(case), int(seed))


def _attend(q, k, v, first):
    """Causal attention in float64: q [n, Hq, D] at positions first.., k and v
    [len, Hkv, D] (rows past a query's position masked)."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    out = torch.empty_like(q)
    pos = first + torch.arange(n, device=q.device)
    mask = torch.arange(k.shape[0], device=q.device)[None, :] > pos[:, None]
    for h in range(hkv):
        kh, vh = k[:, h], v[:, h]
        for j in range(h * (hq // hkv), (h + 1) * (hq // hkv)):
            s = (q[:, j] @ kh.T.contiguous()) / math.sqrt(d)
            out[:, j] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ vh
    return out


def _exact_decode(c, seed):
    x = _decode_inputs(c, seed)
    hkv, d = c["kv_heads"], c["head_dim"]
    k, v, lens, outs = x["k"], x["v"], x["lens"], []
    rows = []
    for b in range(c["batch"]):
        t = np.arange(int(lens[b]) + c["steps"])
        if c["page"]:
            t = x["table"][b, t // c["page"]].astype(np.int64) * c["page"] + t % c["page"]
        else:
            t = b * x["cap"] + t
        rows.append(torch.from_numpy(t).to(DEV))
    for i in range(c["steps"]):
        out = torch.empty(x["q"][i].shape, dtype=torch.float64, device=DEV)
        for b in range(c["batch"]):
            n = int(lens[b]) + i
            k[rows[b][n]] = x["nk"][i, b].reshape(-1).to(k.dtype)
            v[rows[b][n]] = x["nv"][i, b].reshape(-1).to(v.dtype)
            kb = k[rows[b][:n + 1]].double().view(n + 1, hkv, d)
            vb = v[rows[b][:n + 1]].double().view(n + 1, hkv, d)
            qb = x["q"][i, b].double().view(hkv, c["groups"], d)
            s = torch.matmul(qb, kb.permute(1, 2, 0).contiguous()) / math.sqrt(d)
            out[b] = torch.matmul(torch.softmax(s, -1),
                                  vb.permute(1, 0, 2).contiguous()).view(-1, d)
        outs.append(out)
    return {"out": outs, "lens": torch.from_numpy(lens + c["steps"]), "k": None, "v": None}


def _exact_prefill(c, seed):
    x = _prefill_inputs(c, seed)
    hkv, d, cap = c["kv_heads"], c["head_dim"], x["cap"]
    k, v = x["k"].view(-1, cap, hkv, d), x["v"].view(-1, cap, hkv, d)
    out = torch.zeros(x["q"].shape, dtype=torch.float64, device=DEV)
    for b in range(c["batch"]):
        p, n = int(x["start"][b]), int(x["count"][b])
        k[b, p:p + n] = x["nk"][b, :n].to(k.dtype)
        v[b, p:p + n] = x["nv"][b, :n].to(v.dtype)
        out[b, :n] = _attend(x["q"][b, :n].double(), k[b, :p + n].double(),
                             v[b, :p + n].double(), p)
    return {"out": out, "lens": torch.from_numpy(x["start"] + x["count"]), "k": None, "v": None}


def _exact_train(c, seed):
    n, h, d = c["seq"], c["heads"], c["head_dim"]

    def heads(t):
        return t.double().view(c["batch"], n, h, d).transpose(1, 2).contiguous()

    q, k, v, go = (heads(t) for t in _train_inputs(c, seed))
    shape = (c["batch"], h, n)
    o, gq, gk, gv = (torch.empty_like(q) for _ in range(4))
    big, total = (torch.empty(shape, dtype=torch.float64, device=DEV) for _ in range(2))
    mask = torch.ones((n, n), dtype=torch.bool, device=DEV).triu(1)
    sc = 1.0 / math.sqrt(d)
    for b in range(c["batch"]):
        s = (torch.matmul(q[b], k[b].transpose(1, 2).contiguous()) * sc).masked_fill(
            mask, -math.inf)
        big[b] = s.max(-1).values
        e = torch.exp(s - big[b][..., None])
        total[b] = e.sum(-1)
        p = e / total[b][..., None]
        o[b] = torch.matmul(p, v[b])
        ds = p * (torch.matmul(go[b], v[b].transpose(1, 2).contiguous())
                  - (go[b] * o[b]).sum(-1, keepdim=True))
        gv[b] = torch.matmul(p.transpose(1, 2).contiguous(), go[b])
        gq[b] = torch.matmul(ds, k[b]) * sc
        gk[b] = torch.matmul(ds.transpose(1, 2).contiguous(), q[b]) * sc

    def rows(t):
        return t.transpose(1, 2).reshape(c["batch"] * n, h * d)

    def stats(t):
        return t.transpose(1, 2).reshape(-1)

    return {"o": rows(o), "l": stats(total), "m": stats(big), "gq": rows(gq), "gk": rows(gk),
            "gv": rows(gv)}


class _Model64:
    """The model in float64 with a cache of its own, one row per token."""

    def __init__(self, c, seed):
        p = _weights(c, seed)
        self.c = c
        self.emb, self.pe = p["embedding"].double(), p["pos_encoding"].double()
        self.layers = [{k: t.double() for k, t in lp.items()} for lp in p["layers"]]
        self.kv = [None] * c["layers"]

    @staticmethod
    def _norm(x, g, b):
        m = x.mean(-1, keepdim=True)
        return (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + 1e-5) * g + b

    def __call__(self, ids, first, dtype=torch.float64):
        """Logits of ids [B, n] at positions first.. of every row, the cache
        holding first earlier rows; new rows are stored as dtype."""
        c, (b, n), h = self.c, ids.shape, self.c["heads"]
        d = h * c["head_dim"]
        x = self.emb[ids] + self.pe[first:first + n]
        for i, w in enumerate(self.layers):
            y = self._norm(x, w["ln_gamma1"], w["ln_beta1"])
            q, k, v = (torch.matmul(y, w[f]).view(b, n, h, -1)
                       for f in ("attn_wq", "attn_wk", "attn_wv"))
            k, v = k.to(dtype).double(), v.to(dtype).double()
            if self.kv[i] is not None:
                k, v = torch.cat([self.kv[i][0], k], 1), torch.cat([self.kv[i][1], v], 1)
            self.kv[i] = (k, v)
            q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
            s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(c["head_dim"])
            if n > 1:
                mask = (torch.arange(first + n, device=DEV)[None, :]
                        > first + torch.arange(n, device=DEV)[:, None])
                s = s.masked_fill(mask, -math.inf)
            a = torch.matmul(torch.softmax(s, -1), v).transpose(1, 2).reshape(b, n, d)
            x = x + torch.matmul(a, w["attn_wo"])
            y = self._norm(x, w["ln_gamma2"], w["ln_beta2"])
            y = torch.nn.functional.gelu(torch.matmul(y, w["ff_w1"]) + w["ff_b1"],
                                         approximate="tanh")
            x = x + torch.matmul(y, w["ff_w2"]) + w["ff_b2"]
        return torch.matmul(x, self.emb.T.contiguous())


def _exact_forward(c, seed):
    m = _Model64(c, seed)
    ids = torch.from_numpy(_tokens(c, seed, c["batch"], c["tokens"])).to(DEV)
    return m(ids, 0)


def _exact_step(c, seed):
    m = _Model64(c, seed)
    g = _gen(seed + 1)
    dt = _DTYPES[c["dtype"]]
    d = c["heads"] * c["head_dim"]
    for i in range(c["layers"]):
        kv = [torch.randn((c["batch"] * c["context"], d), generator=g, device=DEV).to(dt).double()
              .view(c["batch"], c["context"], c["heads"], -1)[:, :c["fill"]] for _ in range(2)]
        m.kv[i] = tuple(kv)
    ids = torch.from_numpy(_tokens(c, seed, c["steps"], c["batch"])).to(DEV)
    out = [m(ids[i][:, None], c["fill"] + i, dt)[:, 0] for i in range(c["steps"])]
    return {"logits": torch.stack(out), "lens": None, "kv": None}


def _exact_generate(c, seed):
    m, rows = _Model64(c, seed), []
    for prompt in _prompts(c, seed):
        m.kv = [None] * c["layers"]
        ids = torch.tensor([prompt], device=DEV)
        at = 0
        for _ in range(c["new"]):
            logits = m(ids, at)[:, -1]
            at += ids.shape[1]
            ids = logits.argmax(-1, keepdim=True)
        rows.append(logits[0])
    return {"tokens": None, "logits": torch.stack(rows), "kv": None}


def _exact_sample(c, seed):
    return None  # a whole number, not a computed one


_EXACT = {"decode": _exact_decode, "prefill": _exact_prefill, "train": _exact_train,
          "forward": _exact_forward, "step": _exact_step, "generate": _exact_generate,
          "sample": _exact_sample}
