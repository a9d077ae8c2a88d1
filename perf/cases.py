"""The work that an inference engine has these kernels do, as measurable cases.

A case is one engine step or one part of a step, called through the launchers
of redline_amd.kernels as an engine calls them: prefill work is launched
eagerly, decode work is captured once into a HIP graph that each step replays
(every launcher is asynchronous and capturable), except single decode
attention calls, which are launched eagerly.

Kinds:
  decode_step        embedding to fp32 logits for one new token per sequence,
                     INT4 or INT8 weights, over the paged KV cache
  layer_ops          embedding + RMSNorm, then per layer RoPE + KV write,
                     residual add + RMSNorm, SwiGLU
  decode_attention   one decode attention call over a paged cache
  prefill_attention  one causal prefill attention call over a paged cache
  linears            the weight-only projections of some decode layers

Shapes are those of redline_amd.configs; draw() spreads over batch sizes,
context lengths, head layouts, quantisation groups and block sizes, odd and
ragged ones among them.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import redline_amd as ra
from redline_amd import kernels as K
from redline_amd.configs import LLAMA31_8B, QWEN2_7B, TINYLLAMA

_DEV = "cuda"
_EPS = 1e-5
_MODELS = {"tinyllama": TINYLLAMA, "llama": LLAMA31_8B, "qwen2": QWEN2_7B}


def _shape(model):
    m = _MODELS[model]
    return {"hidden": m.hidden, "inter": m.inter, "hq": m.hq, "hkv": m.hkv, "dim": m.head_dim,
            "theta": m.theta}


def _heads(model):
    m = _MODELS[model]
    return {"hq": m.hq, "hkv": m.hkv, "dim": m.head_dim}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # One user chatting with a small model: every launch and every round
        # trip counts (D = 64 heads, INT4 weights, INT8 head).
        {"name": "step_tinyllama_b1", "kind": "decode_step", "batch": 1, "layers": 4, "vocab": 32000,
         "weights": "int4", "group": 128, "kv": "fp16", "block": 16, "ctx_min": 700, "ctx_max": 2000,
         "spread": 1, "bias": False, **_shape("tinyllama")},
        # A loaded server: 32 chats of up to 1024 tokens, INT4 weights and
        # INT8 KV; two of the model's layers and its head.
        {"name": "step_llama_b32", "kind": "decode_step", "batch": 32, "layers": 2, "vocab": 128256,
         "weights": "int4", "group": 128, "kv": "int8", "block": 16, "ctx_min": 64, "ctx_max": 1024,
         "spread": 2, "bias": False, **_shape("llama")},
        # The layer path of a decode step at batch 32, without its products:
        # launch-bound.
        {"name": "layer_ops_decode_b32", "kind": "layer_ops", "layers": 8, "seqs": 32, "new_min": 1,
         "new_max": 1, "past_min": 0, "past_max": 2047, "vocab": 128256, "kv": "fp16",
         "scale16": False, "block": 16, "spread": 3, "bias": False, **_shape("llama")},
        # The layer path of a chunked-prefill step: 4096 rows over FP16 KV.
        {"name": "layer_ops_prefill_4k", "kind": "layer_ops", "layers": 1, "seqs": 4, "new_min": 1024,
         "new_max": 1024, "past_min": 0, "past_max": 3072, "vocab": 128256, "kv": "fp16",
         "scale16": False, "block": 16, "spread": 4, "bias": False, **_shape("llama")},
        # A large prefill step with the QKV bias, INT8 KV and fp16 scales.
        {"name": "layer_ops_prefill_16k", "kind": "layer_ops", "layers": 1, "seqs": 4, "new_min": 4096,
         "new_max": 4096, "past_min": 0, "past_max": 4096, "vocab": 152064, "kv": "int8",
         "scale16": True, "block": 16, "spread": 5, "bias": True, **_shape("qwen2")},
        # Decode attention of a full batch with contexts up to 8192 keys.
        {"name": "decode_attn_b32_8k", "kind": "decode_attention", "batch": 32, "ctx_min": 1,
         "ctx_max": 8192, "kv": "fp16", "scale16": False, "block": 16, "spread": 6,
         **_heads("llama")},
        # A few long documents over INT8 KV, 7 query heads per KV head.
        {"name": "decode_attn_b4_32k_int8", "kind": "decode_attention", "batch": 4, "ctx_min": 16384,
         "ctx_max": 32768, "kv": "int8", "scale16": False, "block": 16, "spread": 7,
         **_heads("qwen2")},
        # Long-context prefill chunks of 4096 tokens at depths up to 12288.
        {"name": "prefill_attn_qwen2_16k", "kind": "prefill_attention", "seqs": 4, "new_min": 4096,
         "new_max": 4096, "past_min": 0, "past_max": 12288, "kv": "fp16", "scale16": False,
         "block": 16, "spread": 8, **_heads("qwen2")},
        # Prefill of four 4096-token prompts into INT8 KV with fp16 scales.
        {"name": "prefill_attn_int8_16k", "kind": "prefill_attention", "seqs": 4, "new_min": 4096,
         "new_max": 4096, "past_min": 0, "past_max": 0, "kv": "int8", "scale16": True,
         "block": 16, "spread": 9, **_heads("llama")},
        # A burst of short chat prompts, ragged lengths, some after a prefix.
        {"name": "prefill_attn_ragged", "kind": "prefill_attention", "seqs": 24, "new_min": 17,
         "new_max": 900, "past_min": 0, "past_max": 700, "kv": "fp16", "scale16": False,
         "block": 16, "spread": 10, **_heads("llama")},
        # The INT4 projections of decode layers at a moderate batch.
        {"name": "linears_int4_b8", "kind": "linears", "batch": 8, "layers": 4, "weights": "int4",
         "group": 128, "bias": False, **_shape("llama")},
        # The INT8 projections of decode layers for one user, QKV bias.
        {"name": "linears_int8_b1", "kind": "linears", "batch": 1, "layers": 2, "weights": "int8",
         "group": 0, "bias": True, **_shape("qwen2")},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_heads(rng):
    dim = rng.choice((64, 128, 128))
    hkv = rng.choice((1, 2, 4, 8))
    return {"hq": hkv * rng.choice((1, 2, 4, 7, 8)), "hkv": hkv, "dim": dim}


def _draw_shape(rng):
    """A known model's layer or a generic one of the same range."""
    if rng.random() < 0.5:
        return _shape(rng.choice(sorted(_MODELS)))
    h = _draw_heads(rng)
    return {"hidden": 128 * rng.randint(8, 48), "inter": 128 * rng.randint(16, 140), **h,
            "theta": rng.choice((1e4, 5e5, 1e6))}


def _draw_once(rng):
    kind = rng.choice(("decode_step", "layer_ops", "decode_attention", "prefill_attention",
                       "prefill_attention", "linears", "linears"))
    kv = rng.choice(("fp16", "int8"))
    c = {"kind": kind, "spread": rng.randrange(1 << 20)}
    if kind in ("decode_step", "linears"):
        c.update(_draw_shape(rng), batch=_log_int(rng, 1, 32), layers=rng.randint(1, 3),
                 weights=rng.choice(("int4", "int4", "int8")), bias=rng.random() < 0.3)
        c["group"] = rng.choice((32, 64, 128, 128)) if c["weights"] == "int4" else 0
    if kind == "decode_step":
        top = _log_int(rng, 32, 4096)
        c.update(vocab=_log_int(rng, 8000, 128256), kv=kv, block=rng.choice((8, 16, 16, 32)),
                 ctx_min=rng.randint(1, top), ctx_max=top)
    elif kind == "layer_ops":
        rows = _log_int(rng, 1, 16384)
        seqs = min(rows, rng.choice((1, 1, 2, 5, 16, 64)))
        new = rows // seqs
        c.update(_draw_shape(rng), layers=1 if rows > 256 else rng.randint(2, 6), seqs=seqs,
                 new_min=max(1, new * 3 // 4), new_max=new, past_min=0,
                 past_max=_log_int(rng, 1, 4096), vocab=_log_int(rng, 8000, 128256), kv=kv,
                 scale16=kv == "int8" and rng.random() < 0.5, block=rng.choice((8, 16, 16, 32)),
                 bias=rng.random() < 0.3)
    elif kind == "decode_attention":
        top = _log_int(rng, 64, 32768)
        c.update(_draw_heads(rng), batch=_log_int(rng, 1, 128), ctx_min=rng.randint(1, top),
                 ctx_max=top, kv=kv, scale16=kv == "int8" and rng.random() < 0.3,
                 block=rng.choice((8, 16, 16, 32)))
    elif kind == "prefill_attention":
        top = _log_int(rng, 24, 8192)
        c.update(_draw_heads(rng), seqs=_log_int(rng, 1, 32), new_min=rng.randint(2, top),
                 new_max=top, past_min=0, past_max=rng.choice((0, _log_int(rng, 16, 8192))), kv=kv,
                 scale16=kv == "int8" and rng.random() < 0.5, block=rng.choice((8, 16, 16, 32)))
    return c


# Bounds of a drawn case, inside the largest listed ones (3.0 GB by
# layer_ops_prefill_16k, 1.9 TFLOP by prefill_attn_qwen2_16k), and of its KV pool.
_MOST_BYTES, _MOST_FLOPS = 1.0e9, 1.2e12
_MOST_KV = 1 << 31


def draw(rng):
    while True:
        c = _draw_once(rng)
        w = work(c)
        kv = 0
        if "ctx_max" in c:
            kv = c["batch"] * c["ctx_max"] * c["hkv"] * c["dim"] * 4
        elif "past_max" in c:
            kv = c["seqs"] * (c["past_max"] + c["new_max"]) * c["hkv"] * c["dim"] * 4
        if w["bytes"] <= _MOST_BYTES and w["flops"] <= _MOST_FLOPS and kv <= _MOST_KV:
            return c


# ------------------------------------------------- sizes, fixed by the case

def _segments(case):
    """(start, new tokens) of each sequence of the step."""
    r = random.Random(case["spread"])
    if "ctx_max" in case:
        return [(r.randint(case["ctx_min"], case["ctx_max"]) - 1, 1) for _ in range(case["batch"])]
    n, lo, hi = case["seqs"], case["past_min"], case["past_max"]
    if case["new_max"] == 1:  # decode rows: contexts at random
        return [(r.randint(lo, hi), 1) for _ in range(n)]
    return [(lo + (hi - lo) * i // max(1, n - 1), r.randint(case["new_min"], case["new_max"]))
            for i in range(n)]


def _projections(case):
    """(name, n, k, takes the bias) of a layer's weight-only products."""
    h, i, d = case["hidden"], case["inter"], case["dim"]
    return [("qkv", (case["hq"] + 2 * case["hkv"]) * d, h, True), ("o", h, case["hq"] * d, False),
            ("gate_up", 2 * i, h, False), ("down", h, i, False)]


def _group(case, k):
    """The largest group up to the case's that divides this K."""
    return math.gcd(case["group"], k)


def _weight_bytes(case, n, k):
    if case["weights"] == "int8":
        return n * k + 2 * n
    return n * k // 2 + 4 * n * (k // _group(case, k))


def _cell_bytes(case):
    """K and V of one token and all KV heads."""
    d, hkv = case["dim"], case["hkv"]
    if case["kv"] == "fp16":
        return 4 * hkv * d
    return hkv * (2 * d + (4 if case.get("scale16") else 8))


def work(case):
    kind, b, f = case["kind"], 0.0, 0.0
    d, hq, hkv = case["dim"], case["hq"], case["hkv"]
    if kind in ("decode_step", "linears"):
        m = case["batch"]
        for name, n, k, _ in _projections(case):
            b += _weight_bytes(case, n, k) + 2 * m * k + 2 * m * (n // 2 if name == "gate_up" else n)
            f += 2 * m * n * k
        b, f = b * case["layers"], f * case["layers"]
    if kind == "decode_step":
        m, h = case["batch"], case["hidden"]
        keys = sum(s + n for s, n in _segments(case))
        layer = keys * _cell_bytes(case) + m * (2 * hq * d * 2 + 2 * _cell_bytes(case) + 16 * h)
        b += case["layers"] * layer + m * 6 * h + case["vocab"] * (h + 2 + 4 * m)
        f += case["layers"] * 4 * d * hq * keys + 2 * m * h * case["vocab"]
    elif kind == "layer_ops":
        rows, h, i = sum(n for _, n in _segments(case)), case["hidden"], case["inter"]
        qkv = (hq + 2 * hkv) * d
        row = 2 * qkv + 2 * hq * d + _cell_bytes(case) + 4 * d + 8 + 8 * h + 6 * i
        b += rows * (case["layers"] * row + 6 * h + 4) + (2 * qkv if case["bias"] else 0)
        f += case["layers"] * rows * (6 * hq * d + 6 * h + 6 * i)
    elif kind == "decode_attention":
        keys = sum(s + n for s, n in _segments(case))
        b += keys * (_cell_bytes(case) + 4 / case["block"]) + case["batch"] * hq * d * 4
        f += 4 * d * hq * keys
    elif kind == "prefill_attention":
        for s, n in _segments(case):
            f += 4 * d * hq * (n * s + n * (n + 1) / 2)
            b += (s + n) * _cell_bytes(case) + n * hq * d * 4
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    """About four times the distance to the 64-bit result, measured over the
    ranges above."""
    kind = case["kind"]
    if kind == "decode_step":  # fp16 roundings travel through the layers
        return {"rel": 6e-3, "max": 0.25, "differ": 5e-3}
    if kind == "layer_ops":  # fp16 activations: about one rounding each
        return {"rel": 1.5e-3, "max": 2e-2, "differ": 2e-3}
    if kind == "linears":
        return {"rel": 1.7e-3, "max": 1e-2}
    return {"rel": 2e-3, "max": 5e-2}  # attention: fp16 probabilities and output


# -------------------------------------------------------------------- inputs

class _Inputs:
    def __init__(self, seed):
        self.g = torch.Generator(device=_DEV).manual_seed(seed)
        self.np = np.random.default_rng(seed)

    def normal(self, shape, std=1.0, mean=0.0):
        return torch.empty(shape, dtype=torch.float16, device=_DEV).normal_(mean, std, generator=self.g)

    def uniform(self, shape, lo, hi, dtype):
        return torch.empty(shape, dtype=dtype, device=_DEV).uniform_(lo, hi, generator=self.g)

    def codes(self, shape, lo, hi, dtype):
        return torch.randint(lo, hi, shape, dtype=dtype, device=_DEV, generator=self.g)


def _batch(case, inp):
    """Metadata of the step from the BatchBuilder, on the GPU: every sequence
    owns its blocks, scattered over the pool."""
    segs, bs = _segments(case), case["block"]
    need = [(s + n + bs - 1) // bs for s, n in segs]
    pool = inp.np.permutation(np.arange(1, sum(need) + 1, dtype=np.int32))
    tokens = sum(n for _, n in segs)
    bb = ra.BatchBuilder(tokens, len(segs), len(segs), max(need), bs, 1)
    at = 0
    for (s, n), k in zip(segs, need):
        bb.add(np.zeros(n, np.int32), s, n, None, pool[at:at + k], mode=ra.LogitsMode.kLast)
        at += k
    meta, shape, lay = bb.write()
    dev = torch.from_numpy(meta[:lay["total_words"]]).to(_DEV)
    return {"meta": dev, "at": lambda name: dev[lay[name]:], "tokens": tokens,
            "blocks": sum(need) + 1, "max_blocks": max(need), "decode_items": shape.num_decode_items,
            "prefill_seqs": shape.num_prefill_seqs, "q_tiles": shape.max_prefill_q_tiles}


def _cache(case, batch, inp, layers):
    """A paged cache filled as earlier steps would have left it."""
    int8 = case["kv"] == "int8"
    c = K.KVCache(layers, batch["blocks"], case["hkv"], case["dim"], case["block"],
                  K.KVDType.kINT8 if int8 else K.KVDType.kFP16,
                  scale_dtype=K.SCALE_F16 if case.get("scale16") else K.SCALE_F32)
    for i in range(layers):
        for t in c.tensors(i)[:2]:
            if int8:
                t.copy_(inp.codes(t.shape, -127, 128, torch.int8))
            else:
                t.normal_(generator=inp.g)
        if int8:
            for t in c.tensors(i)[2:]:
                t.uniform_(0.008, 0.018, generator=inp.g)
    return c


def _weight(case, inp, n, k):
    """A quantised weight [n, k] whose products with unit-variance activations
    have unit variance."""
    if case["weights"] == "int8":
        s = 1.0 / (73.0 * math.sqrt(k))
        return {"n": n, "k": k, "w": inp.codes((n, k), -127, 128, torch.int8),
                "scales": inp.uniform((n,), 0.5 * s, 1.5 * s, torch.float16)}
    s = 1.0 / (4.6 * math.sqrt(k))
    g = _group(case, k)
    scales = inp.uniform((n, k // g), 0.5 * s, 1.5 * s, torch.float16)
    offsets = (scales.float() * -7.5 + inp.uniform((n, k // g), -0.5 * s, 0.5 * s, torch.float32)).half()
    return {"n": n, "k": k, "g": g, "w": inp.codes((n, k // 2), 0, 256, torch.uint8),
            "scales": scales, "offsets": offsets}


def _layer_weights(case, inp):
    p = {}
    for name, n, k, takes_bias in _projections(case):
        p[name] = _weight(case, inp, n, k)
        p[name]["bias"] = inp.normal((n,), 0.02) if takes_bias and case["bias"] else None
    return p


def _linear(p, x, m, y, y_fp32=False):
    if "offsets" in p:
        K.gemv_w4a16(x, m, p["w"], p["scales"], p["offsets"], p["g"], p["bias"], p["n"], p["k"], y, y_fp32)
    else:
        K.gemv_w8a16(x, m, p["w"], p["scales"], p["bias"], p["n"], p["k"], y, y_fp32)


def _gate_up(p, x, m, gate_up, act):
    """silu(gate) * up: in the INT4 product's epilogue, or after the INT8
    product (gate half, then up half)."""
    if "offsets" in p:
        K.gemv_w4a16_swiglu(x, m, p["w"], p["scales"], p["offsets"], p["g"], p["n"], p["k"], act)
    else:
        _linear(p, x, m, gate_up)
        K.silu_and_mul(gate_up, m, p["n"] // 2, act)


def _half(*shape):
    return torch.empty(shape, dtype=torch.float16, device=_DEV)


def _captured(fn):
    """The launches of fn() as a HIP graph (after one eager pass)."""
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph.replay


def _rope_tables(case, batch_case):
    top = max(s + n for s, n in _segments(batch_case))
    cos, sin = ra.rope_cos_sin_tables(case["theta"], case["dim"], top)
    return torch.from_numpy(cos).to(_DEV), torch.from_numpy(sin).to(_DEV)


def _prepare_linears(case, inp, st):
    m = case["batch"]
    st["layers"] = [_layer_weights(case, inp) for _ in range(case["layers"])]
    st["x"] = [{name: inp.normal((m, k)) for name, _, k, _ in _projections(case)}
               for _ in range(case["layers"])]
    gate_up = _half(m, 2 * case["inter"])
    st["out"] = [{name: _half(m, n // 2 if name == "gate_up" else n)
                  for name, n, _, _ in _projections(case)} for _ in range(case["layers"])]

    def step():
        for p, x, y in zip(st["layers"], st["x"], st["out"]):
            _linear(p["qkv"], x["qkv"], m, y["qkv"])
            _linear(p["o"], x["o"], m, y["o"])
            _gate_up(p["gate_up"], x["gate_up"], m, gate_up, y["gate_up"])
            _linear(p["down"], x["down"], m, y["down"])

    st["pass"] = _captured(step)


def _prepare_decode_step(case, inp, st):
    m, h, d, hq, hkv = case["batch"], case["hidden"], case["dim"], case["hq"], case["hkv"]
    L = case["layers"]
    st["batch"] = bt = _batch(case, inp)
    st["cache"] = cache = _cache(case, bt, inp, L)
    st["cos"], st["sin"] = _rope_tables(case, case)
    st["table"] = inp.normal((case["vocab"], h), 0.5)
    st["ids"] = inp.codes((m,), 0, case["vocab"], torch.int32)
    st["norms"] = [inp.normal((h,), 0.1, 1.0) for _ in range(2 * L + 1)]
    st["layers"] = [_layer_weights(case, inp) for _ in range(L)]
    st["head"] = {**_weight({**case, "weights": "int8"}, inp, case["vocab"], h), "bias": None}
    res, x, qkv, att = _half(m, h), _half(m, h), _half(m, (hq + 2 * hkv) * d), _half(m, hq * d)
    gate_up, act, delta = _half(m, 2 * case["inter"]), _half(m, case["inter"]), _half(m, h)
    logits = torch.empty((m, case["vocab"]), dtype=torch.float32, device=_DEV)
    parts = -(-max(s + n for s, n in _segments(case)) // K.kDecodePartitionSize)
    st["ws"] = K.DecodeWorkspace(m, hq, parts, d) if parts > 1 else None
    work_items = K.decode_work(bt["at"]("decode_token"), bt["at"]("decode_seq"), m, parts, st["ws"])
    prms = [K.attention_params(qkv, (hq + 2 * hkv) * d, att, hq, d ** -0.5, cache.layer(i),
                               bt["at"]("block_tables"), bt["max_blocks"], bt["at"]("positions"))
            for i in range(L)]

    def step():
        K.embedding_rmsnorm(st["ids"], st["table"], m, h, st["norms"][0], _EPS, res, x)
        for i, p in enumerate(st["layers"]):
            _linear(p["qkv"], x, m, qkv)
            K.rope_and_write_kv(qkv, bt["at"]("positions"), bt["at"]("slot_mapping"), m, hq, st["cos"],
                                st["sin"], cache.layer(i))
            K.paged_attention_decode(prms[i], work_items)
            _linear(p["o"], att, m, delta)
            K.fused_add_rmsnorm(res, delta, st["norms"][2 * i + 1], m, h, _EPS, x)
            _gate_up(p["gate_up"], x, m, gate_up, act)
            _linear(p["down"], act, m, delta)
            K.fused_add_rmsnorm(res, delta, st["norms"][2 * i + 2], m, h, _EPS, x)
        _linear(st["head"], x, m, logits, True)

    st["before"] = [[t.clone() for t in cache.tensors(i) if t is not None] for i in range(L)]
    st["pass"] = _captured(step)
    st["out"] = {"logits": logits, "residual": res,
                 "cache": [[t for t in cache.tensors(i) if t is not None] for i in range(L)]}
    st["keep"] = (x, qkv, att, gate_up, act, delta, prms, work_items)


def _prepare_layer_ops(case, inp, st):
    h, i, d, hq, hkv, L = (case[k] for k in ("hidden", "inter", "dim", "hq", "hkv", "layers"))
    st["batch"] = bt = _batch(case, inp)
    rows, cols = bt["tokens"], (hq + 2 * hkv) * d
    st["cache"] = cache = _cache(case, bt, inp, L)
    st["cos"], st["sin"] = _rope_tables(case, case)
    st["table"] = inp.normal((case["vocab"], h), 0.5)
    # token frequencies of text are far from even
    st["ids"] = torch.from_numpy(((inp.np.zipf(1.2, rows) - 1) % case["vocab"]).astype(np.int32)).to(_DEV)
    st["norms"] = [inp.normal((h,), 0.1, 1.0) for _ in range(L + 1)]
    st["qkv"] = [inp.normal((rows, cols)) for _ in range(L)]
    st["qkv_bias"] = [inp.normal((cols,), 0.02) if case["bias"] else None for _ in range(L)]
    st["delta"] = [inp.normal((rows, h), 0.3) for _ in range(L)]
    st["gate_up"] = [inp.normal((rows, 2 * i)) for _ in range(L)]
    res, x = _half(rows, h), _half(rows, h)
    act = [_half(rows, i) for _ in range(L)]
    scale = K.SCALE_F16 if case["scale16"] else K.SCALE_F32

    def step():
        K.embedding_rmsnorm(st["ids"], st["table"], rows, h, st["norms"][0], _EPS, res, x)
        for j in range(L):
            if case["bias"] or case["scale16"]:
                K.rope_and_write_kv_ex(st["qkv"][j], bt["at"]("positions"), bt["at"]("slot_mapping"), rows,
                                       hq, st["cos"], st["sin"], cache.layer(j), st["qkv_bias"][j], scale)
            else:
                K.rope_and_write_kv(st["qkv"][j], bt["at"]("positions"), bt["at"]("slot_mapping"), rows,
                                    hq, st["cos"], st["sin"], cache.layer(j))
            K.fused_add_rmsnorm(res, st["delta"][j], st["norms"][j + 1], rows, h, _EPS, x)
            K.silu_and_mul(st["gate_up"][j], rows, i, act[j])

    if rows <= 256:  # decode-sized steps are replayed from a graph
        first = [q.clone() for q in st["qkv"]]
        st["pass"] = _captured(step)
        for q, q0 in zip(st["qkv"], first):
            q.copy_(q0)
    else:
        st["pass"] = step
    # the embedding's own outputs (residual, x) are overwritten by the layers'
    st["out"] = {"residual": res, "x": x, "qkv": st["qkv"], "act": act,
                 "cache": [[t for t in cache.tensors(j) if t is not None] for j in range(L)]}


def _prepare_attention(case, inp, st):
    d, hq, hkv = case["dim"], case["hq"], case["hkv"]
    st["batch"] = bt = _batch(case, inp)
    st["cache"] = cache = _cache(case, bt, inp, 1)
    cols = (hq + 2 * hkv) * d
    st["qkv"] = inp.normal((bt["tokens"], cols), 1.5)  # the q heads of each row are used
    st["out"] = out = _half(bt["tokens"], hq * d)
    prm = K.attention_params(st["qkv"], cols, out, hq, d ** -0.5, cache.layer(0),
                             bt["at"]("block_tables"), bt["max_blocks"], bt["at"]("positions"))
    scale = K.SCALE_F16 if case["scale16"] else K.SCALE_F32
    if case["kind"] == "decode_attention":
        parts = -(-case["ctx_max"] // K.kDecodePartitionSize)
        st["ws"] = K.DecodeWorkspace(bt["decode_items"], hq, parts, d) if parts > 1 else None
        w = K.decode_work(bt["at"]("decode_token"), bt["at"]("decode_seq"), bt["decode_items"], parts, st["ws"])
        plain, ex = K.paged_attention_decode, K.paged_attention_decode_ex
    else:
        w = K.prefill_work(bt["at"]("prefill_seq"), bt["at"]("seq_q_start"), bt["at"]("seq_q_len"),
                           bt["at"]("seq_ctx_len"), bt["prefill_seqs"], bt["q_tiles"])
        plain, ex = K.paged_attention_prefill, K.paged_attention_prefill_ex
    st["pass"] = (lambda: ex(prm, w, scale)) if case["scale16"] else (lambda: plain(prm, w))


def prepare(case, seed):
    inp, st = _Inputs(seed), {}
    {"linears": _prepare_linears, "decode_step": _prepare_decode_step,
     "layer_ops": _prepare_layer_ops, "decode_attention": _prepare_attention,
     "prefill_attention": _prepare_attention}[case["kind"]](case, inp, st)
    return st


def run(state):
    state["pass"]()
    return state["out"]


# ---------------------------------------------------- the results in 64 bits

def _dense(p):
    """The weight's values in float64, [n, k]."""
    if "offsets" not in p:
        return p["w"].double() * p["scales"].double()[:, None]
    w = p["w"].view(p["n"], p["k"] // 2)
    q = torch.stack((w & 15, w >> 4), dim=-1).view(p["n"], p["k"] // p["g"], p["g"]).double()
    return (q * p["scales"].double()[..., None] + p["offsets"].double()[..., None]).view(p["n"], p["k"])


def _linear64(p, x):
    y = x.double() @ _dense(p).t()
    return y if p["bias"] is None else y + p["bias"].double()


def _gate_up64(p, x):
    y = _linear64(p, x)
    if "offsets" in p:  # interleaved rows
        return torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2]
    return _silu_mul64(y)


def _silu_mul64(gate_up):
    half = gate_up.shape[1] // 2
    return torch.nn.functional.silu(gate_up[:, :half]) * gate_up[:, half:]


def _norm64(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + _EPS) * w.double()


def _rope64(x, pos, cos, sin):
    """x [rows, heads, D]: pairs (i, i + D/2)."""
    a, b = x.chunk(2, dim=-1)
    c, s = cos[pos].double()[:, None], sin[pos].double()[:, None]
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def _rows64(t, blocks, cells):
    """Cache rows [keys, hkv, ...] of a sequence in float64."""
    v = t[blocks.long()].transpose(1, 2)  # [nblk, bs, hkv, ...]
    return v.reshape(-1, *v.shape[2:])[:cells].double()


def _keys64(tensors, blocks, ctx):
    k, v, ks, vs = tensors
    k64, v64 = _rows64(k, blocks, ctx), _rows64(v, blocks, ctx)
    if ks is not None:
        k64 = k64 * _rows64(ks, blocks, ctx)[..., None]
        v64 = v64 * _rows64(vs, blocks, ctx)[..., None]
    return k64, v64


def _attend64(q, k64, v64, past):
    """Causal attention of q [n, hq, D] at positions past .. past + n - 1."""
    n, hq, d = q.shape
    group = hq // k64.shape[1]
    out = torch.empty((n, hq, d), dtype=torch.float64, device=q.device)
    key = torch.arange(k64.shape[0], device=q.device)
    for h in range(hq):
        kh, vh = k64[:, h // group].contiguous(), v64[:, h // group].contiguous()
        for r0 in range(0, n, 2048):
            r = torch.arange(r0, min(n, r0 + 2048), device=q.device)
            s = (q[r0:r0 + 2048, h].double() @ kh.t().contiguous()) * d ** -0.5
            s.masked_fill_(key[None] > past + r[:, None], -math.inf)
            out[r0:r0 + 2048, h] = torch.softmax(s, dim=-1) @ vh
    return out.reshape(n, hq * d)


def _tables(case, bt):
    t = bt["at"]("block_tables")[:len(_segments(case)) * bt["max_blocks"]]
    return t.view(-1, bt["max_blocks"])


def _exact_linears(case, st):
    return [{name: (_gate_up64 if name == "gate_up" else _linear64)(p[name], x[name]) for name in p}
            for p, x in zip(st["layers"], st["x"])]


def _exact_attention(case, st):
    bt, d, hq = st["batch"], case["dim"], case["hq"]
    q = st["qkv"][:, :hq * d].reshape(-1, hq, d)
    tables, out, at = _tables(case, bt), [], 0
    for i, (s, n) in enumerate(_segments(case)):
        k64, v64 = _keys64(st["cache"].tensors(0), tables[i], s + n)
        out.append(_attend64(q[at:at + n], k64, v64, s))
        at += n
    return torch.cat(out)


def _exact_decode_step(case, st):
    bt, d, hq, hkv, L = st["batch"], case["dim"], case["hq"], case["hkv"], case["layers"]
    segs, tables = _segments(case), _tables(case, st["batch"])
    pos = bt["at"]("positions")[:case["batch"]].long()
    res = st["table"][st["ids"].long()].double()
    x = _norm64(res, st["norms"][0])
    for i, p in enumerate(st["layers"]):
        qkv = _linear64(p["qkv"], x).view(-1, hq + 2 * hkv, d)
        q, k, v = qkv.split((hq, hkv, hkv), dim=1)
        q, k = _rope64(q, pos, st["cos"], st["sin"]), _rope64(k, pos, st["cos"], st["sin"])
        old = st["before"][i] + [None, None]
        att = []
        for j, (s, n) in enumerate(segs):
            k64, v64 = _keys64(old[:4], tables[j], s + n)
            k64[s], v64[s] = k[j], v[j]
            att.append(_attend64(q[j:j + 1], k64, v64, s))
        res = res + _linear64(p["o"], torch.cat(att))
        x = _norm64(res, st["norms"][2 * i + 1])
        res = res + _linear64(p["down"], _gate_up64(p["gate_up"], x))
        x = _norm64(res, st["norms"][2 * i + 2])
    # the caches hold the rounded rows of the steps before: not compared here
    none = [[None] * len(c) for c in st["out"]["cache"]]
    return {"logits": _linear64(st["head"], x), "residual": res, "cache": none}


def _exact_layer_ops(case, st):
    bt, d, hq, hkv, L = st["batch"], case["dim"], case["hq"], case["hkv"], case["layers"]
    rows = bt["tokens"]
    pos, slot = bt["at"]("positions")[:rows].long(), bt["at"]("slot_mapping")[:rows].long()
    res = st["table"][st["ids"].long()].double()
    out = {"qkv": [], "act": [], "cache": []}
    for j in range(L):
        qkv = st["qkv"][j].double()
        raw = qkv.clone()
        if case["bias"]:
            qkv = qkv + st["qkv_bias"][j].double()
        q, k, v = qkv.view(rows, -1, d).split((hq, hkv, hkv), dim=1)
        raw[:, :hq * d] = _rope64(q, pos, st["cos"], st["sin"]).reshape(rows, -1)
        k = _rope64(k, pos, st["cos"], st["sin"])
        out["qkv"].append(raw)
        tensors = st["cache"].tensors(j)
        bs = case["block"]
        cells = []
        for t, x in zip(tensors, (k, v) if tensors[2] is None else (None, None, k, v)):
            if x is None:  # INT8 codes: whole numbers
                cells.append(None)
                continue
            full = t.double()
            vals = x if tensors[2] is None else x.abs().amax(-1) / 127.0
            full[slot // bs, :, slot % bs] = vals
            cells.append(full)
        out["cache"].append(cells)
        res = res + st["delta"][j].double()
        out["act"].append(_silu_mul64(st["gate_up"][j].double()))
    out["residual"], out["x"] = res, _norm64(res, st["norms"][L])
    return out


def exact(case, seed):
    st = prepare(case, seed)
    return {"linears": _exact_linears, "decode_step": _exact_decode_step,
            "layer_ops": _exact_layer_ops, "decode_attention": _exact_attention,
            "prefill_attention": _exact_attention}[case["kind"]](case, st)
