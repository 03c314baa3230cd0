"""What a program that serves a model through this framework has it do, as cases that can be timed.

A case is a dict of plain values, of one of three kinds:

  decode   one new token per sequence. `step`: the raw projections of the new token go in and the norm, the rotary
           embedding, the cache write and attention run as one call per layer; otherwise attention over rows that are
           in the cache already. `one_call`: all layers in one call.
  prefill  `rows` new positions of one sequence behind `start` rows that the cache holds. By layer: the step before
           attention (norm, rotary embedding, cache write), then attention, one layer after the other, as a forward
           pass calls them. `one_call`: attention of all layers in one call over rows that are in the cache already.
  sample   one token id per row of logits: top-k, softmax, top-p, one draw.

cache / io: element type of the KV cache and of the activations. local: 0, or the window of the local layers, five of
which stand in front of every global one. head_dim is 256 throughout.
"""
import importlib
import math

import numpy as np
import torch

_package = importlib.import_module("litert-lm_amd")
A, S = _package.attn, _package.sampler

D = 256
DEV = "cuda:0"
DTYPE = {"f32": A.F32, "f16": A.F16, "bf16": A.BF16, "i8": A.I8}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8}
SIZE = {"f32": 4, "f16": 2, "bf16": 2, "i8": 1}


def _decode(name, **kw):
    return dict({"name": name, "kind": "decode", "cache": "f16", "io": "f16", "layers": 1, "one_call": False, "step": False,
                 "hq": 8, "hkv": 2, "batch": 1, "context": 4096, "ragged": False, "local": 0, "softcap": 0.0}, **kw)


def _prefill(name, **kw):
    return dict({"name": name, "kind": "prefill", "cache": "bf16", "io": "bf16", "layers": 1, "one_call": False, "hq": 8,
                 "hkv": 2, "rows": 1024, "start": 0, "local": 0, "softcap": 0.0}, **kw)


def _sample(name, **kw):
    return dict({"name": name, "kind": "sample", "batch": 1, "vocab": 262144, "k": 64, "p": 0.95, "temperature": 1.0}, **kw)


def listed():
    return [
        # The smallest call: one layer's step for one token over a float32 cache (the type of the reference's CPU
        # executor), 1,024 tokens of context.
        _decode("decode_one_layer_f32", cache="f32", io="f32", step=True, hq=4, hkv=1, context=1024),
        # One token of a chat through all layers of a 26-layer model in order, at the middle context of the
        # 1,024 + 256 token benchmark protocol: 26 dependent calls.
        _decode("decode_token_26_layers", step=True, layers=26, hq=4, hkv=1, context=1152, local=512),
        # The headline: the caches of 30 layers at 4,096 tokens, one call.
        _decode("decode_30_layers_4096", layers=30, one_call=True),
        # A serving step of one layer: 64 sequences of unequal lengths up to 4,096.
        _decode("decode_64_ragged", batch=64, ragged=True),
        # The same over a quantised cache: 32 full sequences.
        _decode("decode_32_int8", cache="i8", batch=32),
        # A 1,024-token prompt, attention of all 26 layers in one call.
        _prefill("prefill_26_layers_one_call", layers=26, one_call=True, hq=4, hkv=1, local=512),
        # The same prompt as a forward pass runs it: layer by layer.
        _prefill("prefill_26_layers_in_turn", layers=26, hq=4, hkv=1, local=512),
        # A late chunk of a long document, with a length that fits nothing, float32 activations over a half cache.
        _prefill("prefill_late_chunk", cache="f16", io="f32", rows=2047, start=6157),
        # The last 1,024 rows of a 4,096-token sequence over a quantised cache.
        _prefill("prefill_int8", cache="i8", io="bf16", rows=1024, start=3072),
        # A short prompt over a float32 cache.
        _prefill("prefill_short_f32", cache="f32", io="f32", hq=4, hkv=1, rows=300),
        # Token ids for a batch of 64, and for the one sequence of a chat, from a vocabulary of 262,144.
        _sample("sample_64_rows", batch=64),
        _sample("sample_one_row", k=40, p=0.9),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _drawn(case):
    del case["name"]
    return case


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "sample"))
    if kind == "sample":
        return _drawn(_sample("", batch=_log(rng, 1, 64), vocab=_log(rng, 32000, 262144), k=rng.choice((1, 40, 64, 100)),
                              p=rng.choice((0.8, 0.9, 0.95, 1.0)), temperature=rng.choice((0.7, 1.0))))
    cache, io = rng.choice((("f16", "f16"), ("f16", "f16"), ("bf16", "bf16"), ("bf16", "bf16"), ("f16", "f32"),
                            ("bf16", "f32"), ("i8", "f16"), ("i8", "bf16"), ("f32", "f32")))
    hq, hkv = rng.choice(((4, 1), (8, 2), (8, 2), (8, 4), (3, 1)))
    layers = rng.choice((1, 1, 2, 6, 26))
    one_call = layers > 1 and rng.random() < 0.4
    common = {"cache": cache, "io": io, "hq": hq, "hkv": hkv, "local": rng.choice((0, 0, 512)), "layers": layers,
              "softcap": rng.choice((0.0, 0.0, 0.0, 0.0, 50.0)), "one_call": one_call}
    if kind == "decode":
        c = _decode("", batch=_log(rng, 1, 64), context=_log(rng, 64, 8192), ragged=rng.random() < 0.5,
                    step=not one_call and rng.random() < 0.7, **common)
    else:
        c = _prefill("", rows=_log(rng, 16, 2048), start=rng.choice((0, 1)) * _log(rng, 16, 6144), **common)
    most = 4e9 if cache == "f32" else 5e10

    def too_much():
        w = work(c)
        return w["bytes"] > 2e8 or w["flops"] > most

    while too_much() and c["layers"] > 1:
        c["layers"] = (c["layers"] + 1) // 2
        c["one_call"] = one_call and c["layers"] > 1
    while too_much():
        if kind == "decode":
            c["batch"] = max(1, c["batch"] * 2 // 3)
        else:
            c["rows"], c["start"] = max(16, c["rows"] * 2 // 3), c["start"] * 2 // 3
    return _drawn(c)


# ------------------------------------------------------------------------------------------------ what a case is made of
def _windows(c):
    return [c["local"] if (l + 1) % 6 else 0 for l in range(c["layers"])] if c["local"] and c["layers"] > 1 else [c["local"]] * c["layers"]


def _lengths(c):
    """Rows that every sequence attends to, the new one included: 1/16 to all of the context where they are unequal."""
    if not c["ragged"]:
        return [c["context"]] * c["batch"]
    r = np.random.default_rng(c["batch"] * 10007 + c["context"])
    return [int(x) for x in r.integers(max(1, c["context"] // 16), c["context"] + 1, size=c["batch"])]


def _visible(n, window):
    return min(n, window) if window > 0 else n


def work(c):
    if c["kind"] == "sample":
        return {"bytes": c["batch"] * (c["vocab"] * 4 + 8), "flops": c["batch"] * c["vocab"]}
    size, io = SIZE[c["cache"]], SIZE[c["io"]]
    hq, hkv = c["hq"], c["hkv"]
    scales = 2 * hkv * D * 4 if c["cache"] == "i8" else 0
    if c["kind"] == "decode":
        seen = sum(_visible(n, w) for w in _windows(c) for n in _lengths(c))
        new = c["layers"] * c["batch"]
        rows = new * D * (2 * hq * io + (2 * hkv * (io + size) if c["step"] else 0))
        # (the new row of a step comes with the call: it is written, not read)
        return {"bytes": (seen - (new if c["step"] else 0)) * 2 * hkv * D * size + rows + new * scales, "flops": 4 * hq * D * seen}
    n, start = c["rows"], c["start"]
    pairs = sum(_visible(start + i + 1, w) for w in _windows(c) for i in range(n))
    keys = sum(_visible(start + n, w + n - 1 if w else 0) for w in _windows(c))
    nbytes = keys * 2 * hkv * D * size + c["layers"] * (n * 2 * hq * D * io + scales)
    if not c["one_call"]:  # the step before attention: queries read and written once more, keys and values read and written
        nbytes += c["layers"] * n * D * (2 * hq * io + 2 * hkv * (io + size))
    return {"bytes": nbytes, "flops": 4 * hq * D * pairs}


def tolerance(c):
    # About four times what a pass differs by from the same sums in 64 bits: 1.8e-3 (largest 6e-3) for bfloat16
    # activations, which is the rounding of the output, 2.9e-4 to 3.6e-4 (largest 1.8e-3) for half caches, int8 caches
    # and float32 activations over them, 7e-7 (largest 4.5e-6) for a float32 cache. Ids are the same.
    if c["kind"] == "sample":
        return {"rel": 1e-5}
    if c["io"] == "bf16":
        return {"rel": 7e-3, "max": 0.025}
    if c["cache"] == "f32":
        return {"rel": 5e-6, "max": 4e-5}
    return {"rel": 1.4e-3, "max": 8e-3}


# ------------------------------------------------------------------------------------------------ a state and a pass
def _attn(c, tokens, seqs):
    return A.Attn(c["layers"], c["hq"], c["hkv"], D, tokens, seqs, DTYPE[c["cache"]], DTYPE[c["io"]], layer_window=_windows(c),
                  softcap=c["softcap"], stream=torch.cuda.current_stream().cuda_stream)


def _normal(gen, shape, dtype):
    """Unit-variance rows, as keys and queries are behind their norm; an int8 cache holds them at 40 steps a unit."""
    x = torch.randn(shape, generator=gen, device=DEV)
    return (x * 40).round().clamp(-127, 127).to(torch.int8) if dtype == torch.int8 else x.to(dtype)


def _set_scales(at, gen, c, layer, seq):
    s = torch.rand((2, c["hkv"], D), generator=gen, device=DEV) * 0.01 + 0.02
    at.kv_set_scales(layer, seq, s[0].contiguous(), s[1].contiguous())


def _append(at, gen, c, layer, seq, rows):
    shape = (rows, c["hkv"], D)
    if rows:
        at.kv_append(layer, seq, 0, _normal(gen, shape, TORCH[c["cache"]]), _normal(gen, shape, TORCH[c["cache"]]))


def _set_transform(at, seed, layers):
    """Gemma-3-like constants: norms with a learned scale, rotary embedding with a longer base on global layers."""
    r = np.random.default_rng(seed)
    d = np.arange(0, D, 2, dtype=np.float64) / D
    for layer in range(layers):
        theta = 10000.0 if (layer + 1) % 6 else 1000000.0
        w = (r.standard_normal((2, D)) * 0.1).astype(np.float32)
        at.set_layer_transform(layer, norm_q=True, norm_k=True, q_weight=w[0], k_weight=w[1], eps=1e-6, weight_offset=1.0,
                               rope_inv_freq=(theta ** -d).astype(np.float32))


def prepare(c, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    st = {"case": c}
    if c["kind"] == "sample":
        st["logits"] = torch.randn((c["batch"], c["vocab"]), generator=gen, device=DEV) * 3.0
        st["ids"] = torch.zeros((c["batch"],), dtype=torch.int32, device=DEV)
        st["scores"] = torch.zeros((c["batch"],), device=DEV)
        st["sampler"] = S.Sampler(c["k"], c["p"], c["temperature"], c["batch"], seed % 1000003, c["vocab"],
                                  stream=torch.cuda.current_stream().cuda_stream)
        return st
    layers, hq, hkv, io = c["layers"], c["hq"], c["hkv"], TORCH[c["io"]]
    if c["kind"] == "decode":
        n = c["batch"]
        st["lens"] = _lengths(c)
        at = _attn(c, c["context"], n)
        have = [x - 1 for x in st["lens"]] if c["step"] else st["lens"]
        raw = c["step"]
    else:
        n = c["rows"]
        at = _attn(c, c["start"] + n, 1)
        have = [c["start"] + (n if c["one_call"] else 0)]
        raw = not c["one_call"]
    for layer in range(layers):
        for seq, rows in enumerate(have):
            if c["cache"] == "i8":
                _set_scales(at, gen, c, layer, seq)
            _append(at, gen, c, layer, seq, rows)
    st["q"] = _normal(gen, (layers, n, hq, D), io)
    st["out"] = torch.zeros_like(st["q"])
    if raw:
        st["k"], st["v"] = (_normal(gen, (layers, n, hkv, D), io) for _ in range(2))
        _set_transform(at, seed, layers)
        if c["kind"] == "prefill":
            st["rotated"] = torch.zeros_like(st["q"])
    if not c["one_call"]:  # a forward pass holds the tensors of each layer
        st["layer"] = list(zip(*(st[name] for name in ("q", "k", "v", "rotated", "out") if name in st)))
    st["attn"] = at
    return st


def run(st):
    c = st["case"]
    if c["kind"] == "sample":
        st["sampler"].sample_to_id_and_score_buffer(st["logits"], st["ids"], st["scores"])
        return {"ids": st["ids"], "scores": st["scores"]}
    at, q, out = st["attn"], st["q"], st["out"]
    if c["kind"] == "decode":
        lens = st["lens"]
        if c["one_call"]:
            at.decode(0, lens, q, out, n_layers=c["layers"])
        elif c["step"]:
            for layer, (q, k, v, o) in enumerate(st["layer"]):
                at.decode_step(layer, lens, q, k, v, o)
        else:
            for layer, (q, o) in enumerate(st["layer"]):
                at.decode(layer, lens, q, o)
        return out
    n, start = c["rows"], c["start"]
    if c["one_call"]:
        at.prefill(0, 0, start, n, q, out, n_layers=c["layers"])
        return out
    for layer, (q, k, v, rotated, o) in enumerate(st["layer"]):
        at.pre_attention(layer, 0, start, q, k, v, rotated)
        at.prefill(layer, 0, start, n, rotated, o)
    return {"queries": st["rotated"], "out": out}
