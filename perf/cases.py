"""Performance cases: the calls a user of this package makes, over the sizes they are made at.

Six kinds of case, all through the public entry points:

  dense    custom_kernel((a, b, a_scale, b_scale, c)) on operands that are quantised already
  grouped  grouped_kernel(...) on expert-contiguous rows and their row_offsets
  ffn      a dense gated feed-forward block on bf16 tokens: quantise, gate/up with SiLU*mul, quantise, down
  layer    a mixture-of-experts layer on bf16 tokens: top-k, routing, quantise + gather, gate/up with SiLU*mul,
           quantise, down, weighted combine
  quant_a  the activation quantiser
  quant_b  the weight quantiser

Weights are N(0, 0.02) quantised per 128x128 block, activations N(0, 1) per 1x128, as the repository's benchmark
configurations draw them; the square and the small product take N(0, 1) on both sides.
"""
import importlib
import math

import torch

pkg = importlib.import_module("amd-developer-challenge-2025_amd")
moe = importlib.import_module("amd-developer-challenge-2025_amd.moe")
quant = importlib.import_module("amd-developer-challenge-2025_amd.quant")

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # The smallest call: a plumbing-size product, where the launch and the host path count.
        {"name": "dense_256x512x1024", "kind": "dense", "m": 256, "n": 512, "k": 1024, "outliers": 0.0, "b_std": 1.0},
        # The large square product that is the benchmark's default workload.
        {"name": "dense_4096x4096x4096", "kind": "dense", "m": 4096, "n": 4096, "k": 4096, "outliers": 0.0, "b_std": 1.0},
        # A fused attention down-projection over a prefill batch: long K, N off the tile grid, activations with outliers.
        {"name": "dense_4096x2112x7168", "kind": "dense", "m": 4096, "n": 2112, "k": 7168, "outliers": 0.01, "b_std": 0.02},
        # Decode: a batch of 64 tokens against a large weight matrix, bound by reading the weights.
        {"name": "dense_64x18432x7168", "kind": "dense", "m": 64, "n": 18432, "k": 7168, "outliers": 0.0, "b_std": 0.02},
        # The first of the upstream leaderboard's shapes: few output tiles, long K.
        {"name": "dense_1024x1536x7168", "kind": "dense", "m": 1024, "n": 1536, "k": 7168, "outliers": 0.0, "b_std": 0.02},
        # Odd sizes on both sides: rows of a, b and c that start on any byte.
        {"name": "dense_1023x3141x2048", "kind": "dense", "m": 1023, "n": 3141, "k": 2048, "outliers": 0.0, "b_std": 0.02},
        # The grouped gate/up product of a prefill: 4096 tokens, each routed to 8 of 32 experts.
        {"name": "grouped_4096x8of32", "kind": "grouped", "tokens": 4096, "experts": 32, "topk": 8, "n": 4096, "k": 7168, "skew": 0.0},
        # The same experts in decode: 32 tokens, about 8 rows an expert, every expert's weights read once.
        {"name": "grouped_32x8of32", "kind": "grouped", "tokens": 32, "experts": 32, "topk": 8, "n": 4096, "k": 7168, "skew": 0.0},
        # A dense (shared-expert) feed-forward block over a few hundred tokens, an odd number of them.
        {"name": "ffn_250x7168x2048", "kind": "ffn", "tokens": 250, "hidden": 7168, "inter": 2048},
        # Quantising the bf16 activations of a prefill batch.
        {"name": "quant_a_bf16_4096x7168", "kind": "quant_a", "dtype": "bf16", "rows": 4096, "k": 7168},
        # A whole mixture-of-experts layer in prefill: the largest case.
        {"name": "layer_4096x8of32", "kind": "layer", "tokens": 4096, "experts": 32, "topk": 8, "hidden": 7168, "inter": 2048, "skew": 0.0},
        # The same layer in decode.
        {"name": "layer_64x8of32", "kind": "layer", "tokens": 64, "experts": 32, "topk": 8, "hidden": 7168, "inter": 2048, "skew": 0.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size of [lo, hi], spread over its logarithm: half of them on a multiple of 64 where there is one, half wherever they fall."""
    v = _log(rng, lo, hi)
    return max(lo, v // 64 * 64) if v >= 64 and rng.random() < 0.5 else v


def _k(rng, lo, hi):
    return 128 * _log(rng, lo // 128, hi // 128)


def draw(rng):
    kind = rng.choice(("dense", "dense", "dense", "dense", "grouped", "grouped", "ffn", "layer", "layer", "quant_a", "quant_b"))
    if kind == "dense":
        b_std = rng.choice((0.02, 0.02, 1.0))
        return {"kind": kind, "m": _size(rng, 1, 8192), "n": _size(rng, 512, 18432), "k": _k(rng, 256, 7168),
                "outliers": rng.choice((0.0, 0.01)), "b_std": b_std}
    if kind == "ffn":
        return {"kind": kind, "tokens": _size(rng, 1, 4096), "hidden": _k(rng, 1024, 7168), "inter": _k(rng, 512, 4096)}
    if kind in ("quant_a", "quant_b"):
        return {"kind": kind, "dtype": rng.choice(("bf16", "f32")), "rows": _size(rng, 1, 16384), "k": _k(rng, 512, 7168)}
    case = {"kind": kind, "tokens": _size(rng, 1, 4096), "experts": rng.choice((8, 16, 32)), "topk": rng.choice((2, 4, 8)),
            "skew": rng.choice((0.0, 0.5))}
    if kind == "grouped":
        case.update(n=_size(rng, 512, 4096), k=_k(rng, 512, 7168))
    else:
        case.update(hidden=_k(rng, 1024, 7168), inter=_k(rng, 512, 2048))
    return case


def _tokens(gen, rows, k, dtype=torch.bfloat16, outliers=0.0):
    x = torch.randn(rows, k, generator=gen, device=DEVICE)
    if outliers:
        x = torch.where(torch.rand(rows, k, generator=gen, device=DEVICE) < outliers, x * 20.0, x)
    return x.to(dtype)


def _weights(gen, n, k, std=0.02, experts=0):
    """(b, b_scale) as the GEMMs take them: [n, k] K-major, or [experts, n, k] with every expert K-major."""
    if not experts:
        return quant.quantize_b(torch.randn(n, k, generator=gen, device=DEVICE) * std)
    b = torch.empty(experts, k, n, dtype=torch.float8_e4m3fn, device=DEVICE)
    s = torch.empty(experts, k // 128, (n + 127) // 128, device=DEVICE)
    for e in range(experts):
        q, qs = quant.quantize_b(torch.randn(n, k, generator=gen, device=DEVICE) * std)
        b[e].copy_(q.t())
        s[e].copy_(qs.t())
    return b.transpose(1, 2), s.transpose(1, 2)


def _scores(gen, case):
    """Router scores; `skew` makes some experts more popular than others."""
    return torch.randn(case["tokens"], case["experts"], generator=gen, device=DEVICE) \
        + case["skew"] * torch.randn(case["experts"], generator=gen, device=DEVICE)


def _bf16(*shape):
    return torch.zeros(*shape, dtype=torch.bfloat16, device=DEVICE)


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    if kind == "dense":
        a, a_scale = quant.quantize_a(_tokens(gen, case["m"], case["k"], torch.float32, case["outliers"]))
        b, b_scale = _weights(gen, case["n"], case["k"], case["b_std"])
        return {"kind": kind, "data": (a, b, a_scale, b_scale, _bf16(case["m"], case["n"]))}
    if kind == "grouped":
        row_offsets, row_map, _ = moe.route(moe.topk(_scores(gen, case), case["topk"]), case["experts"])
        a, a_scale = quant.quantize_a(_tokens(gen, case["tokens"], case["k"]), row_map)
        b, b_scale = _weights(gen, case["n"], case["k"], experts=case["experts"])
        return {"kind": kind, "data": (a, b, a_scale, b_scale, row_offsets, _bf16(row_map.numel(), case["n"]))}
    if kind in ("quant_a", "quant_b"):
        x = _tokens(gen, case["rows"], case["k"], DTYPES[case["dtype"]])
        return {"kind": kind, "x": x if kind == "quant_a" else x * 0.02}
    tokens, hidden, inter = case["tokens"], case["hidden"], case["inter"]
    experts = case.get("experts", 0)
    rows = tokens * case["topk"] if experts else tokens
    state = {"kind": kind, "x": _tokens(gen, tokens, hidden), "experts": experts,
             "up": _weights(gen, 2 * inter, hidden, experts=experts), "down": _weights(gen, hidden, inter, experts=experts),
             "h": _bf16(rows, inter), "y": _bf16(rows, hidden)}
    if experts:
        scores = _scores(gen, case)
        # the router's weights of the chosen experts, best first as moe.topk orders them
        state.update(scores=scores, topk=case["topk"], gates=torch.softmax(scores.topk(case["topk"], dim=1).values, dim=1))
    return state


def run(state):
    kind = state["kind"]
    if kind == "dense":
        return pkg.custom_kernel(state["data"])
    if kind == "grouped":
        return pkg.grouped_kernel(state["data"])
    if kind in ("quant_a", "quant_b"):
        q, scale = (quant.quantize_a if kind == "quant_a" else quant.quantize_b)(state["x"])
        return q.view(torch.uint8), scale
    x, h, y = state["x"], state["h"], state["y"]
    (up, up_scale), (down, down_scale) = state["up"], state["down"]
    if kind == "ffn":
        a, a_scale = quant.quantize_a(x)
        moe.gate_up_silu((a, up, a_scale, up_scale, None, h))
        a, a_scale = quant.quantize_a(h)
        return h, pkg.custom_kernel((a, down, a_scale, down_scale, y))
    row_offsets, row_map, slot_of = moe.route(moe.topk(state["scores"], state["topk"]), state["experts"])
    a, a_scale = quant.quantize_a(x, row_map)
    moe.gate_up_silu((a, up, a_scale, up_scale, row_offsets, h))
    a, a_scale = quant.quantize_a(h)
    pkg.grouped_kernel((a, down, a_scale, down_scale, row_offsets, y))
    return moe.combine(y, slot_of, state["gates"]), row_offsets, slot_of


def _gemm_bytes(rows, n, k, matrices=1, out=None):
    """Operands, scales and the bf16 result of a product, each once."""
    kb = k // 128
    return rows * k + matrices * n * k + 4 * rows * kb + 4 * matrices * ((n + 127) // 128) * kb + 2 * rows * (n if out is None else out)


def _used(case):
    """Experts that get a row, on average: the others' weights need not be read."""
    e = case["experts"]
    return e * (1.0 - (1.0 - case["topk"] / e) ** case["tokens"])


def work(case):
    kind = case["kind"]
    if kind == "dense":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _gemm_bytes(m, n, k), "flops": 2 * m * n * k}
    if kind == "grouped":
        rows, n, k = case["tokens"] * case["topk"], case["n"], case["k"]
        return {"bytes": _gemm_bytes(rows, n, k, _used(case)), "flops": 2 * rows * n * k}
    if kind in ("quant_a", "quant_b"):
        rows, k = case["rows"], case["k"]
        scales = rows if kind == "quant_a" else (rows + 127) // 128
        return {"bytes": rows * k * ((2 if case["dtype"] == "bf16" else 4) + 1) + 4 * scales * (k // 128), "flops": 0}
    # The steps are calls of their own, so what one hands to the next is written once and read once.
    tokens, hidden, inter = case["tokens"], case["hidden"], case["inter"]
    experts = case.get("experts", 0)
    rows = tokens * case["topk"] if experts else tokens
    used = _used(case) if experts else 1
    quantise = 2 * tokens * hidden + rows * (hidden + 4 * (hidden // 128)) + rows * inter * 3 + 4 * rows * (inter // 128)
    gemms = _gemm_bytes(rows, 2 * inter, hidden, used, inter) + _gemm_bytes(rows, hidden, inter, used)
    route = 4 * tokens * experts + 16 * rows
    combine = 2 * rows * hidden + 2 * tokens * hidden if experts else 0
    return {"bytes": quantise + gemms + route + combine, "flops": 2 * rows * hidden * inter * 3}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quant_a", "quant_b"):
        return "exact"
    # Four times what the path differs by from the same chain with products in 64 bits and the same roundings in between:
    # a product 2.3e-4 (3.4e-4 with outliers; one unit in the last place of bf16, 0.0078, at most), the blocks with a
    # quantisation between two products 1.6e-3 to 2.1e-3 (at most 0.033).
    if kind in ("dense", "grouped"):
        return {"rel": 1.5e-3, "max": 0.032}
    return {"rel": 8e-3, "max": 0.13}
