"""The timed work of this backend, as a program that runs models on it issues it.

Every case goes through the public entry points of `tensorsharp_amd` (the Python twin of the C ABI): single linears at
decode, batched decode and prefill, the grouped launch of a layer's projections, whole decode steps, the fused
attention-output + FFN call of a prompt chunk, GPT-OSS and Qwen-style expert stages, and a linear on host tensors.

A case is a dict of plain values whose `kind` names the family; `draw` gives one more case of the same ranges.  Weights are
N(0, 0.02) in the blocks of their format, activations N(0, 1) fp32, as in the tests and the benchmark.
"""
import math

import numpy as np
import torch

from tensorsharp_amd import HipBasicOps, QuantizedWeight, synth

TYPES = {"f32": 0, "q4_0": 2, "q8_0": 8, "q4_k": 12, "q5_k": 13, "q6_k": 14, "mxfp4": 39}
# block format -> (weights per block, bytes per block)
BLOCKS = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210), "mxfp4": (32, 17)}


def listed():
    return [
        # one token through one linear of a 4B model (Q8_0 file, FFN up): the smallest call, latency counts
        {"name": "linear_decode", "kind": "linear", "type": "q8_0", "rows": 1, "outs": 9728, "ins": 2560},
        # two dozen sequences decoded together, or a speculated run of tokens, through an FFN projection of an 8B model
        {"name": "linear_batch", "kind": "linear", "type": "q4_k", "rows": 24, "outs": 14336, "ins": 4096},
        # a prompt chunk of 512 tokens through the same projection
        {"name": "linear_prefill", "kind": "linear", "type": "q4_k", "rows": 512, "outs": 14336, "ins": 4096},
        # a ragged prompt tail through the projection that mixed files keep in six bits
        {"name": "linear_ragged", "kind": "linear", "type": "q6_k", "rows": 333, "outs": 4096, "ins": 14336},
        # a long prompt through the widest projection of a 27B-class model
        {"name": "linear_long", "kind": "linear", "type": "q8_0", "rows": 2048, "outs": 21504, "ins": 5376},
        # the seven projections of one 8B layer for one token as one grouped launch
        {"name": "group_layer", "kind": "group", "type": "q4_k", "hidden": 4096, "ffn": 14336, "heads": 32, "kv_heads": 8},
        # a decode step: embedding row, layers, final norm and vocabulary projection, at a short and at a long context
        {"name": "model_decode", "kind": "model", "type": "q4_k", "head_type": "q6_k", "layers": 4, "hidden": 4096, "ffn": 14336,
         "heads": 32, "kv_heads": 8, "context": 512, "vocab": 128256, "qk_norm": False},
        {"name": "model_decode_long", "kind": "model", "type": "q8_0", "head_type": "q8_0", "layers": 3, "hidden": 2560, "ffn": 9728,
         "heads": 32, "kv_heads": 8, "context": 4001, "vocab": 32064, "qk_norm": True},
        # attention output projection + FFN of a short prompt, in place on the residual stream
        {"name": "ffn_prompt", "kind": "ffn", "type": "q4_k", "down_type": "q6_k", "rows": 200, "hidden": 4096, "ffn": 14336},
        # GPT-OSS routing + experts: one token, and a prompt chunk
        {"name": "moe_decode", "kind": "moe", "tokens": 1, "experts": 32, "top_k": 4, "hidden": 2880, "ffn": 2880},
        {"name": "moe_prompt", "kind": "moe", "tokens": 256, "experts": 32, "top_k": 4, "hidden": 2880, "ffn": 2880},
        # a linear whose activations and results are host memory, as the managed tensors are
        {"name": "linear_host", "kind": "host", "type": "q4_k", "rows": 32, "outs": 4096, "ins": 4096},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _multiple(rng, low, high, step):
    return max(low, min(high, _log_int(rng, low, high) // step * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "group", "model", "model", "ffn", "moe", "moe", "host"])
    if kind == "linear":
        t = rng.choice(["q4_k", "q4_k", "q8_0", "q8_0", "q6_k", "q5_k", "q4_0", "mxfp4"])
        return {"kind": kind, "type": t, "rows": _log_int(rng, 1, 2048), "outs": _log_int(rng, 1000, 21504),
                "ins": _multiple(rng, 2048, 21504, BLOCKS[t][0]) if rng.random() < 0.5 else rng.choice([2560, 4096, 5120, 14336])}
    if kind == "group":
        kv = rng.choice([2, 4, 8])
        return {"kind": kind, "type": rng.choice(["q4_k", "q8_0", "mxfp4"]), "hidden": _multiple(rng, 1024, 5120, 256),
                "ffn": _multiple(rng, 2048, 17408, 256), "heads": kv * rng.choice([2, 4, 5]), "kv_heads": kv}
    if kind == "model":
        t = rng.choice(["q4_k", "q8_0"])
        kv = rng.choice([2, 4, 8])
        return {"kind": kind, "type": t, "head_type": rng.choice([t, "q6_k"]), "layers": rng.randint(1, 4),
                "hidden": _multiple(rng, 1024, 4096, 256), "ffn": _multiple(rng, 2048, 14336, 256), "heads": kv * rng.choice([2, 4]),
                "kv_heads": kv, "context": _log_int(rng, 1, 4096), "vocab": rng.randint(8000, 64000), "qk_norm": rng.random() < 0.5}
    if kind == "ffn":
        return {"kind": kind, "type": rng.choice(["q4_k", "q8_0"]), "down_type": rng.choice(["q4_k", "q6_k", "q8_0"]),
                "rows": _log_int(rng, 1, 512), "hidden": _multiple(rng, 1024, 4096, 256), "ffn": _multiple(rng, 2048, 14336, 256)}
    if kind == "moe":
        return {"kind": kind, "tokens": _log_int(rng, 1, 512), "experts": rng.choice([16, 32]), "top_k": rng.choice([2, 4]),
                "hidden": _multiple(rng, 1024, 2880, 32), "ffn": _multiple(rng, 1024, 2880, 32)}
    return {"kind": kind, "type": rng.choice(["q4_k", "q8_0", "mxfp4"]), "rows": _log_int(rng, 1, 256),
            "outs": _log_int(rng, 1000, 9728), "ins": _multiple(rng, 1024, 4096, 256)}


class _State:
    pass


def _weight(t, outs, ins, seed):
    """an [outs x ins] weight as raw blocks in device memory"""
    return QuantizedWeight(synth.random_weight(TYPES[t], outs, ins, "cuda", seed), TYPES[t], ins, outs)


def _normal(shape, seed, sigma=1.0, mean=0.0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * sigma + mean


def prepare(case, seed):
    s = _State()
    s.case = case
    s.kind = case["kind"]
    base = seed * 1000
    if s.kind == "linear":
        s.x = _normal((case["rows"], case["ins"]), base)
        s.w = _weight(case["type"], case["outs"], case["ins"], base + 1)
    elif s.kind == "group":
        s.ws = [_weight(case["type"], n, k, base + 1 + i) for i, (n, k) in enumerate(_group_shapes(case))]
        s.xs = [_normal((1, w.ne0), base + 20 + i) for i, w in enumerate(s.ws)]
        s.ys = [torch.empty((1, w.ne1), dtype=torch.float32, device="cuda") for w in s.ws]
        s.pack = HipBasicOps.PrepareGroup(s.ys, s.xs, s.ws)          # a decode loop reuses it for every token
    elif s.kind == "model":
        h, f, d, cap = case["hidden"], case["ffn"], 128, case["context"] + 16
        q, kv = case["heads"] * d, case["kv_heads"] * d
        s.layers = []
        for i in range(case["layers"]):
            b = base + 20 * i
            s.layers.append({
                "qkv": _weight(case["type"], q + 2 * kv, h, b + 1), "o": _weight(case["type"], h, q, b + 2),
                "gate_up": _weight(case["type"], 2 * f, h, b + 3), "down": _weight(case["type"], h, f, b + 4),
                "attn_norm": _normal((h,), b + 5, 0.1, 1.0), "ffn_norm": _normal((h,), b + 6, 0.1, 1.0),
                "q_norm": _normal((d,), b + 7, 0.1, 1.0) if case["qk_norm"] else None,
                "k_norm": _normal((d,), b + 8, 0.1, 1.0) if case["qk_norm"] else None,
                "k_cache": _normal((case["kv_heads"], cap, d), b + 9), "v_cache": _normal((case["kv_heads"], cap, d), b + 10)})
        s.embedding = _weight("q8_0", 4096, h, base + 901)            # rows of the table around the tokens that are met
        s.token = torch.tensor([seed % 4096], dtype=torch.int32, device="cuda")
        s.hidden = torch.empty((1, h), dtype=torch.float32, device="cuda")
        s.norm = _normal((h,), base + 902, 0.1, 1.0)
        s.head = _weight(case["head_type"], case["vocab"], h, base + 903)
        s.logits = torch.empty((1, case["vocab"]), dtype=torch.float32, device="cuda")
    elif s.kind == "ffn":
        h, f = case["hidden"], case["ffn"]
        s.residual_in = _normal((case["rows"], h), base)
        s.residual = torch.empty_like(s.residual_in)
        s.attention = _normal((case["rows"], h), base + 1)
        s.norm = _normal((h,), base + 2, 0.1, 1.0)
        s.out = _weight(case["type"], h, h, base + 3)
        s.gate_up = _weight(case["type"], 2 * f, h, base + 4)
        s.down = _weight(case["down_type"], h, f, base + 5)
    elif s.kind == "moe":
        e, h, f, t = case["experts"], case["hidden"], case["ffn"], case["tokens"]
        s.hidden = _normal((t, h), base)
        s.router = _normal((t, e), base + 1)
        s.gate_up = synth.random_weight(TYPES["mxfp4"], e * 2 * f, h, "cuda", base + 2)
        s.down = synth.random_weight(TYPES["mxfp4"], e * h, f, "cuda", base + 3)
        s.gate_up_bias = _normal((e, 2 * f), base + 4, 0.1)
        s.down_bias = _normal((e, h), base + 5, 0.1)
    else:
        s.x = _normal((case["rows"], case["ins"]), base).cpu().numpy()
        w = _weight(case["type"], case["outs"], case["ins"], base + 1)
        s.w = QuantizedWeight(w.data.cpu().numpy(), w.ggml_type, w.ne0, w.ne1)
        # uploaded once, as a model load does
        HipBasicOps.PreloadQuantizedWeight(s.w.ptr, s.w.ptr, s.w.ggml_type, s.w.ne0, s.w.ne1, s.w.raw_bytes)
        s.keep = _Release(s.w.ptr)
    return s


class _Release:
    """gives the device copy of a preloaded weight back with the state that owns it"""

    def __init__(self, key):
        self.key = key

    def __del__(self):
        HipBasicOps.InvalidateHostBuffer(self.key)


def run(s):
    c = s.case
    if s.kind in ("linear", "host"):
        return HipBasicOps.LinearForward(s.x, s.w)
    HipBasicOps.UseCurrentStream()
    if s.kind == "group":
        HipBasicOps.AddmmQuantGroupDevice(s.pack)
        return s.ys
    if s.kind == "model":
        HipBasicOps.GetRowsQuantDevice(s.hidden, s.embedding, s.token)
        HipBasicOps.TransformerModelDecode(s.hidden, s.layers, c["heads"], c["kv_heads"], 128, c["context"] - 1, 1e-6, 500000.0)
        HipBasicOps.FusedRmsNormMatMulQuant(s.logits, s.hidden, s.norm, 1e-6, s.head)
        return [s.logits, s.hidden, [(L["k_cache"], L["v_cache"]) for L in s.layers]]
    if s.kind == "ffn":
        s.residual.copy_(s.residual_in)                               # the residual stream as the attention left it
        HipBasicOps.FusedOutProjFFN(s.residual, s.attention, s.out, s.norm, 1e-6, s.gate_up, s.down, c["ffn"])
        return s.residual
    weights, ids = HipBasicOps.MoERoute(s.router, c["top_k"])
    out = HipBasicOps.MoEExpertsGptOssForward(s.hidden, ids, weights, s.gate_up, s.gate_up_bias, s.down, s.down_bias, TYPES["mxfp4"],
                                              c["experts"], c["hidden"], c["ffn"])
    return [out, weights, ids]


def _group_shapes(case):
    h, f, q, kv = case["hidden"], case["ffn"], case["heads"] * 128, case["kv_heads"] * 128
    return [(q, h), (kv, h), (kv, h), (h, q), (f, h), (f, h), (h, f)]


def _bytes(t, outs, ins):
    per, size = BLOCKS[t]
    return outs * (ins // per) * size


def work(case):
    kind = case["kind"]
    if kind in ("linear", "host"):
        m, n, k = case["rows"], case["outs"], case["ins"]
        return {"bytes": _bytes(case["type"], n, k) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "group":
        shapes = _group_shapes(case)
        return {"bytes": sum(_bytes(case["type"], n, k) + 4 * (n + k) for n, k in shapes), "flops": sum(2 * n * k for n, k in shapes)}
    if kind == "model":
        h, f, ctx, layers = case["hidden"], case["ffn"], case["context"], case["layers"]
        q, kv = case["heads"] * 128, case["kv_heads"] * 128
        shapes = [(q + 2 * kv, h), (h, q), (2 * f, h), (h, f)]
        cache = 2 * kv * ctx * 4
        return {"bytes": layers * (sum(_bytes(case["type"], n, k) for n, k in shapes) + cache + 8 * h) +
                _bytes(case["head_type"], case["vocab"], h) + _bytes("q8_0", 1, h) + 4 * (case["vocab"] + 2 * h),
                "flops": layers * (sum(2 * n * k for n, k in shapes) + 4 * q * ctx) + 2 * case["vocab"] * h}
    if kind == "ffn":
        m, h, f = case["rows"], case["hidden"], case["ffn"]
        return {"bytes": _bytes(case["type"], h, h) + _bytes(case["type"], 2 * f, h) + _bytes(case["down_type"], h, f) + 4 * (3 * m * h + h),
                "flops": 2 * m * h * (h + 3 * f)}
    t, e, k, h, f = case["tokens"], case["experts"], case["top_k"], case["hidden"], case["ffn"]
    met = e * (1.0 - (1.0 - k / e) ** t)                              # experts that at least one token of a random routing takes
    return {"bytes": int(met * (_bytes("mxfp4", 2 * f, h) + _bytes("mxfp4", h, f) + 4 * (2 * f + h))) + 4 * t * (2 * h + e + 2 * k),
            "flops": 2 * t * k * 3 * h * f}


def tolerance(case):
    """About four times the distance of each path from the same product in 64-bit arithmetic on the dequantized weights:
    fp16 operands with 32-bit sums give 2e-4 to 7e-4 per matmul, activations as pairs of fp6 blocks (MXFP4 on the matrix
    cores) 1.4e-3, 32-bit operands 1e-7; chains of matmuls add up."""
    kind = case["kind"]
    if kind in ("linear", "host"):
        t, one = case["type"], case["rows"] == 1
        if t == "q8_0" and one:
            return {"rel": 1e-5, "max": 1e-4}
        rel = 8e-4 if one else 6e-3 if t == "mxfp4" else 2.8e-3 if t in ("q4_k", "q5_k") else 1.5e-3
    elif kind == "group":
        rel = 1e-5 if case["type"] == "q8_0" else 8e-4
    elif kind == "model":
        rel = 4.5e-3 if case["type"] == "q4_k" else 1e-3
    elif kind == "ffn":
        rel = 5e-3
    else:
        rel = 1.2e-3 if case["tokens"] * case["top_k"] <= 8 else 6e-3
    return {"rel": rel, "max": 8 * rel}
