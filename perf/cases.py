"""The work whose speed is followed from change to change: what an inference stack has this library do for one linear
layer, one MLP block, one expert layer, or one weight tensor that is loaded.

Every case is a dict of plain values; ``op`` says which calls make up one pass:

* ``gemm``      MXFP4 operands that are packed already -> bf16 (``rows`` x ``n`` x ``k``)
* ``nv_linear`` bf16 activations -> NVFP4 quantiser (calibrated per-tensor scale) -> NVFP4 GEMM
* ``mlp``       bf16 activations -> MXFP4 quantiser -> gate+up GEMM with SwiGLU and quantiser -> down projection
* ``moe``       router logits and bf16 activations -> top-2 routing, quantiser, row gather, grouped gate+up with SwiGLU and
                quantiser, grouped down projection, weighted combine
* ``quantize``  fp32 weights -> MXFP4, as a checkpoint is loaded

Activations are N(0, 1) with one channel in a hundred 20 times larger, weights N(0, 0.02).
"""
from __future__ import annotations

import math

import torch

import avelang_amd as ave

WEIGHT_STD = 0.02
MAX_FLOPS = 3.5e12          # of a drawn case; the largest listed one has 11.5e12
MAX_WEIGHTS = 3.2e9         # elements of a drawn case's weights; the listed expert layers have 1.4e9 and 3.2e9


def listed():
    return [
        # one tile of output: the reference's smallest configuration, all launch and latency
        {"name": "gemm_256", "op": "gemm", "rows": 256, "n": 256, "k": 256},
        # decode of 16 sequences, fused gate+up projection: weights read once
        {"name": "gemm_decode_16", "op": "gemm", "rows": 16, "n": 28672, "k": 4096},
        # prefill of 8192 tokens, up projection
        {"name": "gemm_prefill_8192", "op": "gemm", "rows": 8192, "n": 14336, "k": 4096},
        # NVFP4 at a decode batch of 64
        {"name": "nv_decode_64", "op": "nv_linear", "rows": 64, "n": 28672, "k": 4096},
        # NVFP4 down projection over 4096 tokens
        {"name": "nv_prefill_4096", "op": "nv_linear", "rows": 4096, "n": 4096, "k": 14336},
        # one sequence, one token: the latency of a dense block
        {"name": "mlp_decode_1", "op": "mlp", "rows": 1, "hidden": 4096, "inter": 14336},
        # a decode batch of no round size against hidden sizes that no power of two divides
        {"name": "mlp_decode_100", "op": "mlp", "rows": 100, "hidden": 5120, "inter": 13824},
        # a chunk of a prompt, ragged
        {"name": "mlp_chunk_1500", "op": "mlp", "rows": 1500, "hidden": 4096, "inter": 14336},
        # expert layer, 64 sequences decoding: 16 rows an expert
        {"name": "moe_decode_64", "op": "moe", "rows": 64, "experts": 8, "hidden": 4096, "inter": 14336},
        # many small experts on a hidden size whose rows end inside a cache line, mixed prefill and decode
        {"name": "moe_many_1000", "op": "moe", "rows": 1000, "experts": 128, "hidden": 2880, "inter": 2880},
        # expert layer, prefill of 16384 tokens
        {"name": "moe_prefill_16384", "op": "moe", "rows": 16384, "experts": 8, "hidden": 4096, "inter": 14336},
        # one weight tensor of a checkpoint
        {"name": "quantize_weight", "op": "quantize", "rows": 14336, "k": 4096},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _width(rng, low, high, odd_step):
    """A layer width: mostly whole units of 512 or 128 elements, every fifth one only a multiple of ``odd_step``."""
    step = rng.choice((512, 512, 128, 128, odd_step))
    return min(high, max(low, round(_log_int(rng, low, high) / step) * step))


def draw(rng):
    op = rng.choice(("gemm", "gemm", "nv_linear", "nv_linear", "mlp", "mlp", "mlp", "moe", "moe", "quantize"))
    rows = _log_int(rng, 1, 8192)
    if op == "gemm":
        case = {"op": op, "rows": rows, "n": _width(rng, 256, 28672, 8), "k": _width(rng, 256, 16384, 32)}
    elif op == "nv_linear":
        case = {"op": op, "rows": rows, "n": _width(rng, 512, 28672, 8), "k": _width(rng, 512, 16384, 16)}
    elif op == "mlp":
        case = {"op": op, "rows": rows, "hidden": _width(rng, 1024, 8192, 32), "inter": _width(rng, 1024, 16384, 32)}
    elif op == "moe":
        case = {"op": op, "rows": rows, "experts": _log_int(rng, 4, 256), "hidden": _width(rng, 1024, 7168, 32),
                "inter": _width(rng, 512, 14336, 32)}
        while case["experts"] > 4 and 3.0 * case["experts"] * case["hidden"] * case["inter"] > MAX_WEIGHTS:
            case["experts"] = case["experts"] * 3 // 4
    else:
        case = {"op": op, "rows": _width(rng, 256, 28672, 8), "k": _width(rng, 512, 14336, 32)}
        while case["rows"] * case["k"] > 14336 * 8192:
            case["rows"] = case["rows"] * 3 // 4
    while work(case)["flops"] > MAX_FLOPS:
        case["rows"] = case["rows"] * 3 // 4
    return case


def _activations(rows, k, gen):
    x = torch.randn(rows, k, generator=gen, device="cuda")
    x[:, torch.randperm(k, generator=gen, device="cuda")[: max(1, k // 100)]] *= 20.0
    return x


def _weights(rows, k, gen):
    return torch.randn(rows, k, generator=gen, device="cuda") * WEIGHT_STD


def _expert_weights(experts, rows, k, gen):
    packed = torch.empty(experts, rows, k // 2, dtype=torch.uint8, device="cuda")
    scales = torch.empty(experts, rows, k // 32, dtype=torch.uint8, device="cuda")
    for e in range(experts):
        ave.quantize_mxfp4(_weights(rows, k, gen), packed[e], scales[e])
    return packed, scales


def _nv_scale(x):
    return (x.abs().amax().float() / (448.0 * 6.0)).reshape(1)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    op, rows = case["op"], case["rows"]
    s = {"op": op}
    if op == "gemm":
        s["a"] = ave.quantize_mxfp4(_activations(rows, case["k"], gen))
        s["w"] = ave.quantize_mxfp4(_weights(case["n"], case["k"], gen))
    elif op == "nv_linear":
        s["x"] = _activations(rows, case["k"], gen).bfloat16()
        s["x_scale"] = _nv_scale(s["x"])
        w = _weights(case["n"], case["k"], gen)
        s["w_scale"] = _nv_scale(w)
        s["w"] = ave.quantize_nvfp4(w, s["w_scale"])
    elif op == "mlp":
        s["x"] = _activations(rows, case["hidden"], gen).bfloat16()
        s["gate_up"] = ave.quantize_mxfp4(_weights(2 * case["inter"], case["hidden"], gen))
        s["down"] = ave.quantize_mxfp4(_weights(case["hidden"], case["inter"], gen))
    elif op == "moe":
        s["x"] = _activations(rows, case["hidden"], gen).bfloat16()
        s["logits"] = torch.randn(rows, case["experts"], generator=gen, device="cuda")
        s["gate_up"] = _expert_weights(case["experts"], 2 * case["inter"], case["hidden"], gen)
        s["down"] = _expert_weights(case["experts"], case["hidden"], case["inter"], gen)
    else:
        s["x"] = _weights(rows, case["k"], gen)
    return s


def run(s):
    op = s["op"]
    if op == "gemm":
        return ave.gemm_mxfp4_transposed_b(*s["a"], *s["w"])
    if op == "nv_linear":
        codes, scales = ave.quantize_nvfp4(s["x"], s["x_scale"])
        return ave.gemm_nvfp4_transposed_b(codes, scales, s["x_scale"], *s["w"], s["w_scale"])
    if op == "mlp":
        codes, scales = ave.quantize_mxfp4(s["x"])
        h, h_scales = ave.gemm_mxfp4_swiglu_quant_transposed_b(codes, scales, *s["gate_up"])
        return ave.gemm_mxfp4_transposed_b(h, h_scales, *s["down"])
    if op == "moe":
        tokens = s["x"].shape[0]
        rows_of_token = torch.empty(tokens, 2, dtype=torch.int32, device=s["x"].device)
        token_of_row, row_offsets, row_weight = ave.moe_route_top2(s["logits"], rows_of_token=rows_of_token)
        codes, scales = ave.quantize_mxfp4(s["x"])
        a, a_scales = ave.gather_rows_mxfp4(codes, scales, token_of_row)
        h, h_scales = ave.grouped_gemm_mxfp4_swiglu_quant_transposed_b(a, a_scales, *s["gate_up"], row_offsets)
        y = ave.grouped_gemm_mxfp4_transposed_b(h, h_scales, *s["down"], row_offsets)
        out = ave.moe_combine_top2(y, rows_of_token, row_weight, renormalize=True)
        return {"out": out, "row_offsets": row_offsets, "token_of_row": token_of_row, "row_weight": row_weight}
    return ave.quantize_mxfp4(s["x"])


MX, NV = 0.5 + 1.0 / 32, 0.5 + 1.0 / 16     # bytes of one element with its share of a block scale


def work(case):
    op, rows = case["op"], case["rows"]
    if op == "gemm":
        n, k = case["n"], case["k"]
        return {"bytes": MX * (rows + n) * k + 2.0 * rows * n, "flops": 2.0 * rows * n * k}
    if op == "nv_linear":
        n, k = case["n"], case["k"]
        return {"bytes": 2.0 * rows * k + NV * n * k + 2.0 * rows * n, "flops": 2.0 * rows * n * k}
    if op == "mlp":
        h, i = case["hidden"], case["inter"]
        return {"bytes": 4.0 * rows * h + MX * 3 * h * i, "flops": 6.0 * rows * h * i}
    if op == "moe":
        h, i, e = case["hidden"], case["inter"], case["experts"]
        used = e * (1.0 - (1.0 - 1.0 / e) ** (2 * rows))      # experts that get at least one row
        return {"bytes": rows * (4.0 * h + 4.0 * e + 24.0) + MX * 3 * h * i * used, "flops": 12.0 * rows * h * i}
    return {"bytes": (4.0 + MX) * rows * case["k"], "flops": 0.0}


def tolerance(case):
    op = case["op"]
    if op == "quantize":
        return "exact"
    # against the same path in 64 bits the bf16 results are off by 1.66e-3 (2-norm) and by 3.9e-3 at most, for every op
    # (one rounding to bf16); a rounding that falls the other way in the middle of a block shows as less than that
    return {"rel": 6.6e-3, "max": 1.6e-2}
