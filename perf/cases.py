"""The calls that a user of this library makes, as cases that a timing program can prepare, run and compare.

Five kinds of work, each through the public entry points:

    gemm          ``gemm_a8w8_blockscale`` / ``gemm_a8w8_blockscale_bpreshuffle`` on quantised activations
    quant         ``per_group_quant_hip`` (1x128 activation quantiser), scales row-major or transposed
    layer         (add +) RMSNorm + quant, then the projection that reads its result: the step of a decoder layer
    weight_quant  ``weight_per_128x128_quant``: the weights of a layer at load time or after an update
    moe           ``fused_topk`` and ``fused_moe``: the routed expert layer from 16-bit tokens to 16-bit output

Sizes are those of the benchmark (``bench.py``) and of the tests; row counts are what serving brings: one token,
a decode batch, a few hundred rows of mixed prefill and decode, a full prefill chunk.
"""

from __future__ import annotations

import math

import torch

import aiter_amd

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
EPS = 1e-6


def listed():
    return [
        # one token through the smallest projection of the decode set: launch latency and host time
        {"name": "gemm_one_token", "kind": "gemm", "m": 1, "n": 7168, "k": 2048, "dtype": "bf16", "shuffled": False},
        # a decode batch through the widest one, weights shuffled at load time: the weight stream
        {"name": "gemm_decode", "kind": "gemm", "m": 48, "n": 24576, "k": 1536, "dtype": "fp16", "shuffled": True},
        # a few hundred rows, not a round number, through the fused gate + up projection
        {"name": "gemm_mixed", "kind": "gemm", "m": 203, "n": 36864, "k": 7168, "dtype": "bf16", "shuffled": False},
        # a ragged prefill chunk through the low-rank projection whose N is no multiple of 128
        {"name": "gemm_narrow", "kind": "gemm", "m": 3001, "n": 2112, "k": 7168, "dtype": "bf16", "shuffled": True},
        # a full prefill chunk through the fused gate + up projection: the largest call
        {"name": "gemm_prefill", "kind": "gemm", "m": 8192, "n": 36864, "k": 7168, "dtype": "bf16", "shuffled": False},
        # the activations of a double prefill chunk, quantised on their own
        {"name": "quant_prefill", "kind": "quant", "rows": 16384, "cols": 7168, "dtype": "bf16", "transpose": False},
        # a decode step: residual add + norm + quant (scales transposed), then a projection on shuffled weights
        {"name": "layer_decode", "kind": "layer", "rows": 16, "hidden": 7168, "n": 2112, "dtype": "bf16", "add": True,
         "shuffled": True},
        # a prefill step: norm + quant, then a projection on row-major weights
        {"name": "layer_prefill", "kind": "layer", "rows": 2048, "hidden": 7168, "n": 4096, "dtype": "bf16", "add": False,
         "shuffled": False},
        # the gate + up weights of a layer, quantised when they are loaded
        {"name": "weights_load", "kind": "weight_quant", "n": 36864, "k": 7168, "dtype": "bf16"},
        # the expert layer: a small decode batch, a batch of mixed prefill and decode, a prefill chunk
        {"name": "moe_decode", "kind": "moe", "tokens": 16, "experts": 256, "topk": 8, "dim": 7168, "inter": 256, "dtype": "bf16"},
        {"name": "moe_mixed", "kind": "moe", "tokens": 500, "experts": 256, "topk": 8, "dim": 7168, "inter": 256, "dtype": "bf16"},
        {"name": "moe_prefill", "kind": "moe", "tokens": 8192, "experts": 256, "topk": 8, "dim": 7168, "inter": 256,
         "dtype": "bf16"},
    ]


# the largest listed cases bound what a drawn one may cost
_GEMM_MOST = 8192 * 36864 * 7168
_MOE_MOST = 8192 * 8 * 7168 * 256


def _spread(rng, low, high, step=1):
    """A multiple of `step` in [low, high], evenly spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "quant", "layer", "weight_quant", "moe", "moe", "moe"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "gemm":
        n, k = _spread(rng, 576, 36864, 64), _spread(rng, 512, 7168, 128)
        return {"kind": kind, "m": _spread(rng, 1, min(8192, _GEMM_MOST // (n * k))), "n": n, "k": k, "dtype": dtype,
                "shuffled": rng.random() < 0.5}
    if kind == "quant":
        return {"kind": kind, "rows": _spread(rng, 1, 16384), "cols": _spread(rng, 1024, 7168, 128), "dtype": dtype,
                "transpose": rng.random() < 0.5}
    if kind == "layer":
        return {"kind": kind, "rows": _spread(rng, 1, 8192), "hidden": _spread(rng, 1024, 8192, 128),
                "n": _spread(rng, 576, 8192, 64), "dtype": dtype, "add": rng.random() < 0.5, "shuffled": rng.random() < 0.5}
    if kind == "weight_quant":
        return {"kind": kind, "n": _spread(rng, 576, 36864, 64), "k": _spread(rng, 512, 7168, 128), "dtype": dtype}
    experts, topk = rng.choice([(256, 8), (256, 8), (128, 8), (64, 6), (40, 6), (32, 5), (8, 2)])
    dim, inter = _spread(rng, 1024, 7168, 256), rng.choice([128, 256, 256, 384, 512, 1024])
    most = min(8192, _MOE_MOST // (topk * dim * inter))
    return {"kind": kind, "tokens": _spread(rng, 1, most), "experts": experts, "topk": topk, "dim": dim, "inter": inter,
            "dtype": dtype}


def _randn(gen, *shape, scale=1.0):
    return torch.randn(*shape, generator=gen, device=gen.device) * scale


def _activations(gen, rows, cols, dtype):
    """N(0, 1) with one channel in a hundred 50 times as large: what reaches a projection in practice."""
    x = _randn(gen, rows, cols)
    loud = torch.randperm(cols, generator=gen, device=gen.device)[: max(1, cols // 100)]
    x[:, loud] *= 50.0
    return x.to(dtype)


def _weights(gen, n, k, scale=0.02):
    """[n, k] fp8 codes and their 128 x 128 scales, in pieces that keep the 16-bit original small."""
    codes = torch.empty(n, k, dtype=aiter_amd.dtypes.fp8, device=gen.device)
    scales = torch.empty((n + 127) // 128, k // 128, dtype=torch.float32, device=gen.device)
    step = 32768
    for lo in range(0, n, step):
        part = _randn(gen, min(step, n - lo), k, scale=scale).bfloat16()
        c, s = aiter_amd.weight_per_128x128_quant(part)
        codes[lo:lo + step], scales[lo // 128:lo // 128 + s.shape[0]] = c, s
    return codes, scales


def _shuffled(codes):
    return aiter_amd.shuffle_weight(codes, layout=(16, 16))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, kind = DTYPES[case["dtype"]], case["kind"]
    state = dict(case, dtype=dtype)
    if kind == "gemm":
        x = _activations(gen, case["m"], case["k"], dtype)
        state["xq"], state["xs"] = aiter_amd.per_group_quant_hip(x, transpose_scale=case["shuffled"])
        wq, state["ws"] = _weights(gen, case["n"], case["k"])
        state["wq"] = _shuffled(wq) if case["shuffled"] else wq
    elif kind == "quant":
        state["x"] = _activations(gen, case["rows"], case["cols"], dtype)
    elif kind == "layer":
        rows, hidden = case["rows"], case["hidden"]
        state["x"] = _activations(gen, rows, hidden, dtype)
        state["residual"] = _randn(gen, rows, hidden).to(dtype) if case["add"] else None
        state["residual_out"] = torch.empty_like(state["x"]) if case["add"] else None
        state["gain"] = (torch.rand(hidden, generator=gen, device=gen.device) + 0.5).to(dtype)
        state["xq"] = torch.empty(rows, hidden, dtype=aiter_amd.dtypes.fp8, device=gen.device)
        state["xs"] = torch.empty(rows, hidden // 128, dtype=torch.float32, device=gen.device)
        wq, state["ws"] = _weights(gen, case["n"], hidden)
        state["wq"] = _shuffled(wq) if case["shuffled"] else wq
    elif kind == "weight_quant":
        state["w"] = _randn(gen, case["n"], case["k"], scale=0.02).to(dtype)
    else:
        tokens, experts, dim, inter = case["tokens"], case["experts"], case["dim"], case["inter"]
        state["x"] = _randn(gen, tokens, dim).to(dtype)
        # some experts are liked better than others, as trained routers do
        state["gating"] = _randn(gen, tokens, experts) + _randn(gen, 1, experts, scale=0.5)
        w1, s1 = _weights(gen, experts * 2 * inter, dim, scale=0.1)
        w2, s2 = _weights(gen, experts * dim, inter, scale=0.1)
        state["w1"], state["w1_scale"] = _shuffled(w1.view(experts, 2 * inter, dim)), s1.view(experts, -1)
        state["w2"], state["w2_scale"] = _shuffled(w2.view(experts, dim, inter)), s2.view(experts, -1)
    return state


def _project(s, xq, xs):
    if s["shuffled"]:
        return aiter_amd.gemm_a8w8_blockscale_bpreshuffle(xq, s["wq"], xs, s["ws"], s["dtype"])
    return aiter_amd.gemm_a8w8_blockscale(xq, s["wq"], xs, s["ws"], s["dtype"])


def run(state):
    s = state
    kind = s["kind"]
    if kind == "gemm":
        return _project(s, s["xq"], s["xs"])
    if kind == "quant":
        return aiter_amd.per_group_quant_hip(s["x"], transpose_scale=s["transpose"])
    if kind == "layer":
        if s["add"]:
            aiter_amd.rmsnorm2d_fwd_with_add_dynamicquant(s["xq"], s["x"], s["residual"], s["residual_out"], s["xs"], s["gain"],
                                                          EPS, 0, 128, s["shuffled"])
            return s["xq"], s["xs"], s["residual_out"], _project(s, s["xq"], s["xs"])
        aiter_amd.rmsnorm2d_fwd_with_dynamicquant(s["xq"], s["x"], s["xs"], s["gain"], EPS, 0, 128, s["shuffled"])
        return s["xq"], s["xs"], _project(s, s["xq"], s["xs"])
    if kind == "weight_quant":
        return aiter_amd.weight_per_128x128_quant(s["w"])
    weights, ids = aiter_amd.fused_topk(s["x"], s["gating"], s["topk"], True)
    out = aiter_amd.fused_moe(s["x"], s["w1"], s["w2"], weights, ids, w1_scale=s["w1_scale"], w2_scale=s["w2_scale"])
    return weights, ids, out


def _gemm_work(m, n, k):
    return m * k + 4 * m * (k // 128) + n * k + 4 * -(-n // 128) * (k // 128) + 2 * m * n, 2 * m * n * k


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        moved, flops = _gemm_work(case["m"], case["n"], case["k"])
    elif kind == "quant":
        n = case["rows"] * case["cols"]
        moved, flops = 3 * n + 4 * n // 128, 3 * n  # magnitude, maximum, quotient
    elif kind == "layer":
        rows, hidden = case["rows"], case["hidden"]
        n = rows * hidden
        moved, flops = _gemm_work(rows, case["n"], hidden)
        # the codes and scales between the two are written and read; the residual stream is read and written
        moved += 3 * n + 4 * n // 128 + 2 * hidden + (4 * n if case["add"] else 0)
        flops += (8 if case["add"] else 7) * n  # add, square, sum, two products, magnitude, maximum, quotient
    elif kind == "weight_quant":
        n = case["n"] * case["k"]
        moved, flops = 3 * n + 4 * -(-case["n"] // 128) * (case["k"] // 128), 3 * n
    else:
        tokens, experts, topk, dim, inter = (case[v] for v in ("tokens", "experts", "topk", "dim", "inter"))
        hit = experts * (1.0 - (1.0 - topk / experts) ** tokens)  # experts that an even routing meets
        per_expert = 3 * inter * dim + 4 * 3 * -(-inter // 128) * (dim // 128)
        moved = hit * per_expert + tokens * (4 * dim + 4 * experts + 8 * topk)
        flops = 6 * tokens * topk * dim * inter + 3 * tokens * experts
    return {"bytes": float(moved), "flops": float(flops)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quant", "weight_quant"):
        return "exact"
    # About four times the largest error seen against the same arithmetic in 64 bits (relative, largest): bf16 1.7e-3 and
    # 4.1e-3, fp16 2.1e-4 and 7.7e-4.  It is the rounding of the stored result, and does not depend on the size.
    if kind in ("gemm", "layer"):
        return {"rel": 7e-3, "max": 0.016} if case["dtype"] == "bf16" else {"rel": 9e-4, "max": 0.003}
    # The activation product is rounded to fp8 between the two matrix products: where the order of a sum moves a value
    # across a rounding boundary, a token's row moves by a sixteenth of that value's share.  Seen: 2.6e-3 and 4.9e-2.
    return {"rel": 1.05e-2, "max": 0.2}
