"""The work that users of this package have it do, as cases that can be timed.

A case is a dict of plain values.  `listed()` gives the ones that stand for the package's use, `draw(rng)` one more of
the same ranges, `prepare(case, seed)` the tensors a caller holds before the call, `run(state)` one pass through the
public ops, `work(case)` the bytes and operations that pass cannot do without, `tolerance(case)` how far apart two
correct implementations may be.

Kinds (m = weight rows, n = tokens, k = reduction length, as everywhere in this package):
  matmul     one projection: ops.matmul, or ops.matmul_fused where an epilogue is named
  blockwise  one projection whose weights have a scale per `block` elements: ops.matmul_blockwise
  multi      Q, K and V kept as separate weights and multiplied in one call: ops.matmul_multi
  layer      the four projections of a decoder layer in the order a model calls them: QKV, attention out with the
             residual added, gate+up with SiLU-mul, down with the residual added (attention itself, between the first
             two, is the caller's; its result is an input here)
  grouped    the experts of a mixture on tokens sorted by expert: ops.matmul_grouped
  dequant    packed weights to fp16: ops.dequant
  quantize   fp16 weights to packed ones, as at model load: ops.quantize
"""
import math
import random

import torch

from tuna_amd import ops, synth
from tuna_amd._lib import EPILOGUE_RESIDUAL, EPILOGUE_SILU_MUL
from tuna_amd.quantize import nf4_codebook

MOST_FLOPS = 8e11   # of a drawn case; the largest listed one does 8.7e11
MOST_BYTES = 4e8    # of a drawn case; the largest listed one moves 4.3e8


def listed():
    return [
        # a chat with one user: the smallest projection of a 7B model, one token; the launch is most of it
        {"name": "matmul_1_token", "kind": "matmul", "m": 4096, "n": 1, "k": 4096, "epilogue": "none"},
        # a small decode batch: the QKV projection of the benchmark's headline
        {"name": "matmul_16_tokens", "kind": "matmul", "m": 6144, "n": 16, "k": 4096, "epilogue": "none"},
        # an odd decode batch on a down projection whose k has few factors of two
        {"name": "matmul_37_tokens", "kind": "matmul", "m": 5120, "n": 37, "k": 13824, "epilogue": "none"},
        # decode of a 70B model at the paper's batch: 428 MB of weights per layer
        {"name": "layer_70b_16_tokens", "kind": "layer", "hidden": 8192, "qkv": 10240, "ffn": 28672, "n": 16},
        # decode of a 7B model with a full batch
        {"name": "layer_7b_64_tokens", "kind": "layer", "hidden": 4096, "qkv": 6144, "ffn": 14336, "n": 64},
        # prefill of a 7B model: a prompt is as long as it is
        {"name": "layer_7b_2000_tokens", "kind": "layer", "hidden": 4096, "qkv": 6144, "ffn": 14336, "n": 2000},
        # the usual quantization block, decode and prefill
        {"name": "blockwise_16_tokens", "kind": "blockwise", "m": 28672, "n": 16, "k": 4096, "block": 64},
        {"name": "blockwise_777_tokens", "kind": "blockwise", "m": 4096, "n": 777, "k": 14336, "block": 128},
        # gate+up of eight experts, two per token: a decode batch of 64 and a prefill of 2048 tokens
        {"name": "grouped_decode", "kind": "grouped", "m": 28672, "groups": 8, "k": 4096, "n": 128, "route": 1},
        {"name": "grouped_prefill", "kind": "grouped", "m": 14336, "groups": 8, "k": 4096, "n": 4096, "route": 2},
        # weights handed to a library that wants fp16, and a checkpoint quantized while it loads
        {"name": "dequant_down", "kind": "dequant", "m": 4096, "k": 14336, "block": 0},
        {"name": "quantize_gate", "kind": "quantize", "m": 14336, "k": 4096, "block": 64},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo, hi, unit):
    """A width between lo and hi in multiples of `unit`, spread over the logarithm."""
    return max(1, round(_log_int(rng, lo, hi) / unit)) * unit


def _unit(rng):
    """Most models' widths are multiples of 128; some are only multiples of 64, and the ops take any multiple of 8."""
    return rng.choice((128, 128, 128, 128, 128, 64, 64, 8, 8))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            return case


def _draw(rng):
    kind = rng.choice(("matmul", "matmul", "matmul", "matmul", "layer", "layer", "blockwise", "blockwise", "grouped",
                       "grouped", "multi", "dequant", "quantize"))
    n = _log_int(rng, 1, 4096)
    if kind == "matmul":
        unit = _unit(rng)
        return {"kind": kind, "m": _width(rng, 1024, 57344, unit), "n": n, "k": _width(rng, 1024, 28672, unit),
                "epilogue": rng.choice(("none", "none", "residual", "silu_mul"))}
    if kind == "layer":
        unit = rng.choice((128, 128, 256))
        hidden = _width(rng, 1024, 8192, unit)
        kv = rng.choice((hidden, hidden // 4, 1024))
        return {"kind": kind, "hidden": hidden, "qkv": hidden + 2 * kv, "ffn": _width(rng, 2 * hidden, 5 * hidden, 128),
                "n": min(n, 2000)}
    if kind == "blockwise":
        return {"kind": kind, "m": _width(rng, 1024, 57344, 64), "n": n, "k": _width(rng, 1024, 28672, 256),
                "block": rng.choice((64, 64, 128))}
    if kind == "grouped":
        groups = rng.choice((8, 8, 16, 64))
        return {"kind": kind, "m": _width(rng, 1024, 28672, 128), "groups": groups, "k": _width(rng, 1024, 14336, 128),
                "n": _log_int(rng, 8, 8192), "route": rng.randrange(1 << 20)}
    if kind == "multi":
        hidden = _width(rng, 1024, 8192, 256)
        return {"kind": kind, "hidden": hidden, "kv": rng.choice((hidden, hidden // 4, 1024)), "n": _log_int(rng, 1, 64)}
    unit = _unit(rng)
    if kind == "dequant":
        unit = max(unit, 64)
        return {"kind": kind, "m": _width(rng, 1024, 28672, unit), "k": _width(rng, 1024, 14336, unit),
                "block": rng.choice((0, 0, 64))}
    unit = max(unit, 64)
    return {"kind": kind, "m": _width(rng, 1024, 28672, unit), "k": _width(rng, 1024, 14336, unit),
            "block": rng.choice((0, 64, 64))}


def token_offsets(case):
    """Rows of x per expert: each token picks experts independently, some experts are liked up to twice as well."""
    rng = random.Random(case["route"])
    like = [rng.uniform(1.0, 2.0) for _ in range(case["groups"])]
    counts = [0] * case["groups"]
    for e in rng.choices(range(case["groups"]), like, k=case["n"]):
        counts[e] += 1
    offs = [0]
    for c in counts:
        offs.append(offs[-1] + c)
    return offs


def _weights(m, k, seed, dev, block=0):
    q, s = synth.make_weights_torch(m, k, seed, dev)
    if block:
        g = torch.Generator(device=dev)
        g.manual_seed(seed + 104729)
        s = torch.empty((m, k // block), dtype=torch.float32, device=dev).uniform_(0.005, 0.02, generator=g)
    return q, s


def _out(n, m, dev):
    return torch.empty((n, m), dtype=torch.float16, device=dev)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    kind = case["kind"]
    code = nf4_codebook(dev)
    if kind in ("matmul", "blockwise"):
        m, n, k = case["m"], case["n"], case["k"]
        q, s = _weights(m, k, seed, dev, case.get("block", 0))
        x = synth.make_x_torch(n, k, seed, dev)
        if kind == "blockwise":
            return kind, (x, q, s, code, _out(n, m, dev), m, n, k, case["block"])
        if case["epilogue"] == "none":
            return kind, (x, q, s, code, _out(n, m, dev), m, n, k)
        if case["epilogue"] == "residual":
            residual = synth.make_x_torch(n, m, seed + 1, dev)
            return "fused", (x, q, s, code, _out(n, m, dev), m, n, k, EPILOGUE_RESIDUAL, residual)
        return "fused", (x, q, s, code, _out(n, m // 2, dev), m, n, k, EPILOGUE_SILU_MUL)
    if kind == "layer":
        h, qkv, ffn, n = case["hidden"], case["qkv"], case["ffn"], case["n"]
        x = synth.make_x_torch(n, h, seed, dev)
        attn = synth.make_x_torch(n, h, seed + 1, dev)
        shapes = ((qkv, h), (h, h), (2 * ffn, h), (h, ffn))
        w = [_weights(m, k, 4 * seed + i, dev) for i, (m, k) in enumerate(shapes)]
        o = [_out(n, c, dev) for c in (qkv, h, ffn, h)]
        return kind, (x, attn, code, w, o, h, qkv, ffn, n)
    if kind == "multi":
        h, n = case["hidden"], case["n"]
        x = synth.make_x_torch(n, h, seed, dev)
        problems = []
        for i, m in enumerate((h, case["kv"], case["kv"])):
            q, s = _weights(m, h, 3 * seed + i, dev)
            problems.append((x, q, s, code, _out(n, m, dev), m, n, h))
        return kind, problems
    if kind == "grouped":
        m, groups, k, n = case["m"], case["groups"], case["k"], case["n"]
        q, s = _weights(groups * m, k, seed, dev)
        x = synth.make_x_torch(n, k, seed, dev)
        return kind, (x, q, s, code, _out(n, m, dev), m, groups, k, token_offsets(case))
    m, k, block = case["m"], case["k"], case["block"] or None
    if kind == "dequant":
        q, s = _weights(m, k, seed, dev, case["block"])
        return kind, (q, s, code, _out(m, k, dev), m, k, block)
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    w = (torch.randn(m, k, dtype=torch.float32, device=dev, generator=g) * 0.02).half()
    return kind, (w, code, block)


def run(state):
    kind, a = state
    if kind == "matmul":
        ops.matmul(*a)
        return a[4]
    if kind == "fused":
        ops.matmul_fused(*a)
        return a[4]
    if kind == "blockwise":
        ops.matmul_blockwise(*a)
        return a[4]
    if kind == "layer":
        x, attn, code, w, (o_qkv, o_h, o_ff, o_y), h, qkv, ffn, n = a
        ops.matmul(x, w[0][0], w[0][1], code, o_qkv, qkv, n, h)
        ops.matmul_fused(attn, w[1][0], w[1][1], code, o_h, h, n, h, EPILOGUE_RESIDUAL, x)
        ops.matmul_fused(o_h, w[2][0], w[2][1], code, o_ff, 2 * ffn, n, h, EPILOGUE_SILU_MUL)
        ops.matmul_fused(o_ff, w[3][0], w[3][1], code, o_y, h, n, ffn, EPILOGUE_RESIDUAL, o_h)
        return a[4]
    if kind == "multi":
        ops.matmul_multi(a)
        return [p[4] for p in a]
    if kind == "grouped":
        ops.matmul_grouped(*a)
        return a[4]
    if kind == "dequant":
        q, s, code, o, m, k, block = a
        ops.dequant(q, s, code, o, m, k, block_size=block)
        return o
    w, code, block = a
    q, absmax, _ = ops.quantize(w, code, block_size=block)
    return q, absmax


def _gemm(m, n, k, block=0):
    """(bytes, flops): packed weights, scales and x in, out out."""
    return m * k / 2 + 4 * m * (k // block if block else 1) + 2 * n * k + 2 * n * m, 2.0 * m * n * k


def work(case):
    kind = case["kind"]
    if kind in ("matmul", "blockwise"):
        m, n, k = case["m"], case["n"], case["k"]
        b, f = _gemm(m, n, k, case.get("block", 0))
        b += {"residual": 2 * n * m, "silu_mul": -n * m}.get(case.get("epilogue"), 0)
    elif kind == "layer":
        h, qkv, ffn, n = case["hidden"], case["qkv"], case["ffn"], case["n"]
        params = (qkv + h) * h + 3 * ffn * h
        # in: weights, scales, x and the attention's result; out: the four results
        b = params / 2 + 4 * (qkv + 2 * h + 2 * ffn) + 2 * n * (2 * h) + 2 * n * (qkv + 2 * h + ffn)
        f = 2.0 * n * params
    elif kind == "multi":
        h, n = case["hidden"], case["n"]
        rows = h + 2 * case["kv"]
        b, f = _gemm(rows, n, h)
    elif kind == "grouped":
        m, k, n = case["m"], case["k"], case["n"]
        offs = token_offsets(case)
        active = sum(hi > lo for lo, hi in zip(offs, offs[1:]))
        b = active * (m * k / 2 + 4 * m) + 2 * n * (k + m)
        f = 2.0 * m * n * k
    else:
        m, k, block = case["m"], case["k"], case["block"]
        b = 2.5 * m * k + 4 * m * (k // block if block else 1)
        f = 0
    return {"bytes": b, "flops": f}


def tolerance(case):
    # codes, scales and decoded weights are a function of the inputs, rounding included
    if case["kind"] in ("dequant", "quantize"):
        return "exact"
    # fp16 results of 32-bit sums in any order; in a layer the next projection reads the rounded result
    return {"rel": 1e-3}
