"""The workloads whose speed this package is judged by, each as a program that uses it would run it.

A case is a dict of plain values. `op` names the path:

  fp8_gemm     operands already in e4m3: one dispatch_fp8_gemm per weight matrix
  fp8_linear   bf16 activations: per-tensor quantization, then one dispatch_fp8_gemm per weight matrix
  bf16_gemm    one dispatch_bf16_gemm per weight matrix
  mxfp4_linear bf16 activations: dispatch_mxfp4_quantize_rows, then one dispatch_mxfp4_gemm per weight matrix
  moe_mxfp4    one mixture-of-experts layer with MXFP4 weights (activations MXFP4 or MXFP8, plain SiLU or
               biases and clamped SwiGLU), from router logits to the layer's output
  moe_fp8blk   one mixture-of-experts layer with block-scaled e4m3 weights and group-limited sigmoid routing,
               from e4m3 or bf16 activations, with or without the expert that every token passes through

`weights` of the GEMM paths is the number of weight matrices that a pass takes the same activations through:
a token's pass through a model touches each matrix once, so a decode step never finds one in a cache.
"""
from __future__ import annotations

import math

import torch

import hipkittens_amd as hk

tk = hk.tk_kernel

_GEMM_OPS = ("fp8_gemm", "fp8_linear", "bf16_gemm", "mxfp4_linear")
_GEMM_FLOPS = 2.0 * 8192 ** 3   # the largest GEMM that is drawn: the listed square one
_MOE_MXFP4_FLOPS = 6.0 * 16384 * 4 * 2880 * 2880
_MOE_FP8BLK_FLOPS = 6.0 * 8192 * 8 * 7168 * 2048


def listed():
    return [
        # the smallest square of the benchmark's sweep: one launch of a few microseconds, latency and host time count
        {"name": "fp8_gemm_1024", "op": "fp8_gemm", "M": 1024, "N": 1024, "K": 1024, "weights": 1},
        # the headline: a compute-bound prefill or training GEMM
        {"name": "fp8_gemm_8192", "op": "fp8_gemm", "M": 8192, "N": 8192, "K": 8192, "weights": 1},
        # gate and up projection of a dense MLP for a chunk of 200 prompt tokens (or 200 decoding sequences)
        {"name": "fp8_linear_chunk", "op": "fp8_linear", "M": 200, "N": 14336, "K": 4096, "weights": 2},
        # down projections of eight layers for four decoding sequences: the weights stream from HBM
        {"name": "bf16_gemm_decode", "op": "bf16_gemm", "M": 4, "N": 4096, "K": 14336, "weights": 8},
        # a ragged prompt through one projection
        {"name": "bf16_gemm_prefill", "op": "bf16_gemm", "M": 3001, "N": 4096, "K": 4096, "weights": 1},
        # 64 decoding sequences through sixteen projections, activations quantized once
        {"name": "mxfp4_linear_decode", "op": "mxfp4_linear", "M": 64, "N": 8192, "K": 8192, "weights": 16},
        # a 4096-token prompt through a projection of the MoE models' hidden size (rows of 90 scale bytes)
        {"name": "mxfp4_linear_prefill", "op": "mxfp4_linear", "M": 4096, "N": 2880, "K": 2880, "weights": 1},
        # decode step of the GPT-OSS-like layer: four sequences, sixteen experts at most
        {"name": "moe_mxfp4_decode", "op": "moe_mxfp4", "T": 4, "H": 2880, "I": 2880, "E": 128, "k": 4,
         "act": "mxfp4", "swiglu": True},
        # a batch of 1000 tokens with MXFP8 activations: every expert has a few rows, the weights dominate
        {"name": "moe_mxfp4_batch", "op": "moe_mxfp4", "T": 1000, "H": 2880, "I": 2880, "E": 128, "k": 4,
         "act": "mxfp8", "swiglu": False},
        # prefill of 16384 tokens: 512 rows an expert, compute bound
        {"name": "moe_mxfp4_prefill", "op": "moe_mxfp4", "T": 16384, "H": 2880, "I": 2880, "E": 128, "k": 4,
         "act": "mxfp4", "swiglu": True},
        # decode step of the DeepSeek-V3-like layer with its shared expert, 16 sequences
        {"name": "moe_fp8blk_decode", "op": "moe_fp8blk", "T": 16, "H": 7168, "I": 2048, "E": 256, "k": 8,
         "x": "bf16", "shared": True},
        # prefill of 8192 tokens through the same layer's routed experts
        {"name": "moe_fp8blk_prefill", "op": "moe_fp8blk", "T": 8192, "H": 7168, "I": 2048, "E": 256, "k": 8,
         "x": "e4m3", "shared": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, of):
    return min(hi, max(lo, -(-_log_int(rng, lo, hi) // of) * of))


def _draw_gemm(rng, op):
    while True:
        M = _log_int(rng, 1, 8192)
        # whole tiles mostly; widths like a vocabulary's can be anything
        N = _multiple(rng, 512, 32768, rng.choice((64, 64, 16, 1)))
        K = _multiple(rng, 512, 16384, rng.choice((256, 256, 32)))
        width = {"bf16_gemm": 2.0, "mxfp4_linear": 0.53125}.get(op, 1.0)
        size = N * K * width
        # a decode step or a small chunk goes through many matrices, a prompt is counted by the matrix
        weights = max(1, min(32, int(512e6 / size))) if M <= 512 and rng.random() < 0.75 else 1
        if size <= 512e6 and 2.0 * M * N * K * weights <= _GEMM_FLOPS:
            return {"op": op, "M": M, "N": N, "K": K, "weights": weights}


def _draw_moe_mxfp4(rng):
    while True:
        T = _log_int(rng, 1, 16384)
        H, I = (2880, 2880) if rng.random() < 0.5 else (_multiple(rng, 1024, 4096, 64), _multiple(rng, 512, 4096, 64))
        E, k = rng.choice(((128, 4), (128, 8), (64, 4), (32, 4), (32, 2)))
        case = {"op": "moe_mxfp4", "T": T, "H": H, "I": I, "E": E, "k": k,
                "act": "mxfp8" if rng.random() < 0.3 else "mxfp4", "swiglu": rng.random() < 0.5}
        if 6.0 * T * k * H * I <= _MOE_MXFP4_FLOPS:
            return case


def _draw_moe_fp8blk(rng):
    while True:
        T = _log_int(rng, 1, 8192)
        H, I = (7168, 2048) if rng.random() < 0.5 else (_multiple(rng, 1024, 7168, 128), _multiple(rng, 512, 2048, 128))
        E, k = rng.choice(((256, 8), (128, 8), (64, 6), (64, 4)))
        shared = rng.random() < 0.5
        case = {"op": "moe_fp8blk", "T": T, "H": H, "I": I, "E": E, "k": k,
                "x": "bf16" if shared or rng.random() < 0.5 else "e4m3", "shared": shared}
        if 6.0 * T * (k + shared) * H * I <= _MOE_FP8BLK_FLOPS:
            return case


def draw(rng):
    op = rng.choice(_GEMM_OPS + ("moe_mxfp4", "moe_mxfp4", "moe_fp8blk"))
    if op == "moe_mxfp4":
        return _draw_moe_mxfp4(rng)
    if op == "moe_fp8blk":
        return _draw_moe_fp8blk(rng)
    return _draw_gemm(rng, op)


# ------------------------------------------------------------------------------------------ preparation
def _randn(g, *shape):
    return torch.randn(*shape, device=g.device, generator=g)


def _prepare_gemm(case, g):
    op, M, N, K, n = case["op"], case["M"], case["N"], case["K"], case["weights"]
    dev = g.device
    x = _randn(g, M, K).to(torch.bfloat16)
    s = {"op": op, "x": x, "C": [torch.empty((M, N), dtype=torch.bfloat16, device=dev) for _ in range(n)]}
    if op == "bf16_gemm":
        s["W"] = [(_randn(g, N, K) * 0.02).to(torch.bfloat16) for _ in range(n)]
        size = tk.bf16_gemm_workspace_bytes(M, N, K)
    elif op == "mxfp4_linear":
        s["W"] = [hk.quant.quantize_mxfp4(_randn(g, N, K) * 0.02) for _ in range(n)]
        s["xq"] = torch.empty((M, K // 2), dtype=torch.uint8, device=dev)
        s["xs"] = torch.empty((M, -(-K // 256) * 8), dtype=torch.uint8, device=dev)   # rows of whole 8 bytes
        size = tk.mxfp4_gemm_workspace_bytes(M, N, K)
    else:
        s["W"] = [hk.quant.quantize_fp8_per_tensor(_randn(g, N, K) * 0.02) for _ in range(n)]
        if op == "fp8_gemm":
            s["xq"], s["x_scale"] = hk.quant.quantize_fp8_per_tensor(x)
        size = tk.fp8_gemm_workspace_bytes(M, N, K)
    s["ws"] = torch.empty(size, dtype=torch.uint8, device=dev) if size else None
    return s


def _prepare_moe_mxfp4(case, g):
    T, H, I, E, k = (case[n] for n in ("T", "H", "I", "E", "k"))
    dev = g.device

    def experts(rows, cols):
        """[E, rows, cols] weights quantized expert by expert, scale rows padded to whole 8 bytes."""
        packed = torch.empty((E, rows, cols // 2), dtype=torch.uint8, device=dev)
        scales = torch.empty((E, rows, -(-cols // 256) * 8), dtype=torch.uint8, device=dev)
        for e in range(E):
            packed[e], s = hk.quant.quantize_mxfp4(_randn(g, rows, cols) * 0.02)
            scales[e] = hk.quant.pad_scales(s)
        return packed, scales

    W = tk.MoeMxfp4ShuffledWeights.from_plain(*experts(2 * I, H), *experts(H, I), interleaved=case["swiglu"])
    options = {"act_format": case["act"]}
    if case["swiglu"]:
        options.update(bias13=_randn(g, E, 2 * I) * 0.1, bias2=_randn(g, E, H) * 0.1, activation="swiglu_oai")
    # trained routers do not spread tokens evenly: some experts are asked for two or three times as often
    logits = _randn(g, T, E) + 0.3 * _randn(g, E)
    return {"op": "moe_mxfp4", "x": _randn(g, T, H).to(torch.bfloat16), "logits": logits, "W": W, "k": k,
            "options": options, "y": torch.empty((T, H), dtype=torch.bfloat16, device=dev),
            "ws": torch.empty(tk.moe_mxfp4_workspace_bytes(T, H, I, E, k, act_format=case["act"]), dtype=torch.uint8,
                              device=dev)}


def _fp8blk_weights(g, E, H, I):
    dev = g.device
    w13 = torch.empty((E, 2 * I, H), dtype=torch.float8_e4m3fn, device=dev)
    s13 = torch.empty((E, 2 * I // 128, H // 128), dtype=torch.float32, device=dev)
    w2 = torch.empty((E, H, I), dtype=torch.float8_e4m3fn, device=dev)
    s2 = torch.empty((E, H // 128, I // 128), dtype=torch.float32, device=dev)
    for e in range(E):
        w13[e], s13[e] = hk.quant.quantize_fp8_blocks(_randn(g, 2 * I, H) * 0.02, 128, 128)
        w2[e], s2[e] = hk.quant.quantize_fp8_blocks(_randn(g, H, I) * 0.02, 128, 128)
    return tk.MoeFp8BlkShuffledWeights.from_plain(w13, s13, w2, s2)


def _prepare_moe_fp8blk(case, g):
    T, H, I, E, k = (case[n] for n in ("T", "H", "I", "E", "k"))
    dev = g.device
    x = _randn(g, T, H).to(torch.bfloat16)
    # the selection bias is what a trained router uses to keep its experts evenly loaded
    s = {"op": "moe_fp8blk", "k": k, "x": x, "logits": _randn(g, T, E), "bias": _randn(g, E) * 0.05,
         "W": _fp8blk_weights(g, E, H, I), "y": torch.empty((T, H), dtype=torch.bfloat16, device=dev),
         "ws": torch.empty(tk.moe_fp8blk_workspace_bytes(T, H, I, E, k), dtype=torch.uint8, device=dev)}
    s["quantize"] = case["shared"]
    if case["shared"] or case["x"] == "e4m3":
        s["xq"] = torch.empty((T, H), dtype=torch.float8_e4m3fn, device=dev)
        s["xs"] = torch.empty((T, H // 128), dtype=torch.float32, device=dev)
    if case["shared"]:
        s["shared"] = _fp8blk_weights(g, 1, H, I)
        s["y_shared"] = torch.empty((T, H), dtype=torch.bfloat16, device=dev)
        s["ws_shared"] = torch.empty(tk.moe_fp8blk_workspace_bytes(T, H, I, 1, 1), dtype=torch.uint8, device=dev)
    elif case["x"] == "e4m3":
        tk.dispatch_fp8_quantize_rows_1x128(x, s["xq"], s["xs"])
    return s


def prepare(case, seed):
    g = torch.Generator(device=torch.device("cuda", torch.cuda.current_device())).manual_seed(seed)
    if case["op"] == "moe_mxfp4":
        return _prepare_moe_mxfp4(case, g)
    if case["op"] == "moe_fp8blk":
        return _prepare_moe_fp8blk(case, g)
    return _prepare_gemm(case, g)


# ------------------------------------------------------------------------------------------ one pass
def _run_gemm(s):
    op, ws = s["op"], s["ws"]
    if op == "bf16_gemm":
        for w, c in zip(s["W"], s["C"]):
            tk.dispatch_bf16_gemm(s["x"], w, c, workspace=ws)
    elif op == "mxfp4_linear":
        tk.dispatch_mxfp4_quantize_rows(s["x"], s["xq"], s["xs"])
        for (w, ws_b), c in zip(s["W"], s["C"]):
            tk.dispatch_mxfp4_gemm(s["xq"], s["xs"], w, ws_b, c, workspace=ws)
    else:
        xq, scale = (s["xq"], s["x_scale"]) if op == "fp8_gemm" else hk.quant.quantize_fp8_per_tensor(s["x"])
        for (w, w_scale), c in zip(s["W"], s["C"]):
            tk.dispatch_fp8_gemm(xq, w, c, scale, w_scale, workspace=ws)
    return s["C"]


def _run_moe_fp8blk(s):
    x, xs, add = s["x"], None, None
    if s["quantize"]:
        tk.dispatch_fp8_quantize_rows_1x128(s["x"], s["xq"], s["xs"])
    if "xq" in s:
        x, xs = s["xq"], s["xs"]
    if "shared" in s:
        add = s["y_shared"]
        tk.dispatch_moe_fp8blk_shared_expert(x, xs, s["shared"], None, None, None, add, s["ws_shared"])
    tk.dispatch_moe_fp8blk(x, xs, s["logits"], s["bias"], s["W"], None, None, None, s["y"], s["k"], 8, 4, 2.5,
                           s["ws"], y_add=add)
    return s["y"]


def run(state):
    if state["op"] == "moe_mxfp4":
        tk.dispatch_moe_mxfp4(state["x"], state["logits"], state["W"], None, None, None, state["y"], state["k"],
                              state["ws"], **state["options"])
        return state["y"]
    if state["op"] == "moe_fp8blk":
        return _run_moe_fp8blk(state)
    return _run_gemm(state)


# ------------------------------------------------------------------------------------------ what it takes
def work(case):
    """Bytes and operations of one pass: every input, weight and output once; of a layer of experts the weights
    of those that T tokens with k choices each are expected to touch."""
    if case["op"] in _GEMM_OPS:
        M, N, K, n = case["M"], case["N"], case["K"], case["weights"]
        w = {"bf16_gemm": 2.0, "mxfp4_linear": 0.53125}.get(case["op"], 1.0)
        x = 1.0 if case["op"] == "fp8_gemm" else 2.0
        return {"bytes": x * M * K + n * (w * N * K + 2.0 * M * N), "flops": 2.0 * M * N * K * n}
    T, H, I, E, k = (case[n] for n in ("T", "H", "I", "E", "k"))
    touched = E * (1.0 - (1.0 - k / E) ** T)
    if case["op"] == "moe_mxfp4":
        weights, extra = touched * (3.0 * H * I * 0.53125 + (4.0 * (2 * I + H) if case["swiglu"] else 0.0)), 0
        x = 2.0
    else:
        extra = 1 if case["shared"] else 0
        weights = (touched + extra) * 3.0 * H * I * (1.0 + 4.0 / 16384)
        x = 2.0 if case["x"] == "bf16" else 1.0 + 4.0 / 128
    return {"bytes": weights + T * H * (x + 2.0) + 4.0 * T * E, "flops": 6.0 * T * (k + extra) * H * I}


def tolerance(case):
    """About four times what the paths differ from 64-bit sums (rounded to bf16 like theirs) on these inputs. GEMM:
    2-norm 2.4e-4 (e4m3: the matrix unit keeps fewer bits of its products than fp32; the others less), single
    elements one unit in the last place of bf16. The layers of experts round their hidden activations to 4 or 8 bits between
    their two GEMMs, where a sum that lies at a tie may fall to either side: 2-norm 2.4e-4 / 1.1e-3 / 2.1e-3
    (MXFP4 / MXFP8 / block-scaled e4m3), single elements up to 0.01 / 0.015 / 0.021 of the output's root mean square."""
    if case["op"] == "moe_mxfp4":
        return {"rel": 4.5e-3, "max": 0.06}
    if case["op"] == "moe_fp8blk":
        return {"rel": 8e-3, "max": 0.09}
    return {"rel": 1e-3, "max": 0.03}
