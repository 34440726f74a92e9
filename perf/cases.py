"""Workloads of the Q8_0 path, for timing it and for comparing its results.

Each case is one call (or one short chain of calls) that a program running a Q8_0 model
makes through ``llmengine_amd.capi``: the Linears of a decode step and of a prompt, on raw
GGUF bytes and on weights re-tiled at load time, their fused forms, the Q8_0 MatMul, the
embedding gather, and the picks from the logits.  Shapes are those of the benchmark
(Llama-7B and Qwen2.5-0.5B Linears) or generic ones of the same ranges; values have the
benchmark's distributions: activations N(0, 1), quants uniform on [-127, 127], binary16
scales |N(0, 1)| * 0.02 / 127, ids uniform over the table.
"""
from __future__ import annotations

import math

import torch

from llmengine_amd import capi

BLOCK = 32         # elements of a Q8_0 block
BLOCK_BYTES = 34   # binary16 scale + 32 int8 quants
GEMM_TOKENS = 64   # from here on the Linear and the MatMul round both operands to bf16

MAX_MNK = 2048 * 4096 * 11008  # no drawn case takes more products than the largest listed one


def listed():
    return [
        # Smallest call of a decode step: the fused q/k/v projection of a 0.5B model, one
        # sequence, fp32 biases.  Launch latency and a handful of row groups.
        {"name": "qwen_qkv_m1", "kind": "multi", "M": 1, "N": 896, "N2": 128, "N3": 128,
         "K": 896, "layout": "tiled", "bias": "f32"},
        # One-sequence decode of a 7B model: the fused q/k/v projection, bound by the weights.
        {"name": "llama_qkv_m1", "kind": "multi", "M": 1, "N": 4096, "N2": 4096, "N3": 4096,
         "K": 4096, "layout": "tiled", "bias": "none"},
        # A small decode batch on the GGUF bytes as a loader copies them, long rows.
        {"name": "llama_down_raw_m4", "kind": "linear", "M": 4, "N": 4096, "K": 11008,
         "layout": "raw", "bias": "none"},
        # Feed-forward front of a decode batch of eight: gate, up and SwiGLU in one call.
        {"name": "llama_swiglu_m8", "kind": "swiglu", "M": 8, "N": 11008, "K": 4096,
         "layout": "tiled"},
        # A serving batch of 32 sequences, one token each.
        {"name": "llama_qkv_m32", "kind": "linear", "M": 32, "N": 12288, "K": 4096,
         "layout": "tiled", "bias": "none"},
        # A short prompt of odd length through an attention output projection, bf16 bias.
        {"name": "llama_o_m77", "kind": "linear", "M": 77, "N": 4096, "K": 4096,
         "layout": "tiled", "bias": "bf16"},
        # The benchmark's prefill: 512 tokens on the GGUF bytes.
        {"name": "llama_gate_raw_m512", "kind": "linear", "M": 512, "N": 11008, "K": 4096,
         "layout": "raw", "bias": "none"},
        # A long prompt on tiled weights, the largest case.
        {"name": "llama_down_m2048", "kind": "linear", "M": 2048, "N": 4096, "K": 11008,
         "layout": "tiled", "bias": "none"},
        # End of a greedy decode step: the 152k-row head, then the argmax of its logits.
        {"name": "qwen_head_greedy_m1", "kind": "head", "M": 1, "N": 151936, "K": 896,
         "layout": "tiled"},
        # Sampling for eight sequences: the 40 likeliest tokens of each logits row.
        {"name": "qwen_top40_m8", "kind": "top", "M": 8, "N": 151936, "k": 40,
         "temperature": 0.8},
        # A prompt batch's embedding rows: 8 sequences of 512 tokens.
        {"name": "qwen_embedding_4096", "kind": "embedding", "M": 4096, "N": 151936, "K": 896,
         "layout": "raw"},
        # The Q8_0 MatMul (blocks along N) on a decode batch of eight.
        {"name": "matmul_m8", "kind": "matmul", "M": 8, "N": 4096, "K": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "multi", "swiglu", "swiglu",
                       "matmul", "matmul", "embedding", "top", "head"])
    layout = rng.choice(["tiled", "tiled", "raw"])
    if kind == "top":
        return {"kind": kind, "M": rng.randint(1, 16), "N": _log_int(rng, 4000, 152000),
                "k": rng.randint(1, 128), "temperature": round(rng.uniform(0.5, 1.5), 2)}
    if kind == "embedding":
        return {"kind": kind, "M": _log_int(rng, 1, 4096), "N": _log_int(rng, 4000, 151936),
                "K": BLOCK * rng.randint(16, 28), "layout": layout}
    if kind == "head":
        return {"kind": kind, "M": rng.randint(1, 8), "N": _log_int(rng, 32000, 151936),
                "K": BLOCK * rng.randint(16, 28), "layout": layout}
    K = BLOCK * _log_int(rng, 16, 344)
    if kind == "matmul":
        M, N = _log_int(rng, 1, 512), BLOCK * _log_int(rng, 16, 344)
        return {"kind": kind, "M": M, "N": N, "K": K}
    # Outputs per call; about half of them whole 16-row groups, as model sizes mostly are.
    M, N = _log_int(rng, 1, 2048), _log_int(rng, 500, 12288)
    if rng.random() < 0.5:
        N = max(512, N // 128 * 128)
    if kind == "swiglu":
        N = min(N, 11008)
    parts = {"linear": 1, "multi": 3, "swiglu": 2}[kind]
    N = min(N, 88_000_000 // (parts * K))
    M = max(1, min(M, MAX_MNK // (parts * N * K), 8_000_000 // (parts * N)))
    case = {"kind": kind, "M": M, "N": N, "K": K, "layout": layout}
    if kind == "linear":
        case["bias"] = rng.choice(["none", "none", "f32", "bf16"])
    if kind == "multi":
        case["N2"] = case["N3"] = max(1, N // rng.choice([1, 1, 4, 7]))
        case["bias"] = rng.choice(["none", "f32"])
    return case


def _outputs(case):
    """Sizes of a Linear's weights: one, the q/k/v three, or the gate/up pair."""
    if case["kind"] == "multi":
        return [case["N"], case["N2"], case["N3"]]
    return [case["N"], case["N"]] if case["kind"] == "swiglu" else [case["N"]]


def _q8_0(gen, rows, cols):
    """Raw Q8_0 bytes of a [rows, cols] tensor with the benchmark's distributions."""
    blocks = rows * (cols // BLOCK)
    raw = torch.empty((blocks, BLOCK_BYTES), dtype=torch.uint8, device="cuda")
    z = torch.randn(blocks, 1, generator=gen, device="cuda")
    raw[:, :2] = (z.abs_() * (0.02 / 127.0)).half().view(torch.uint8)
    raw[:, 2:] = torch.randint(-127, 128, (blocks, BLOCK), generator=gen, device="cuda",
                               dtype=torch.int8).view(torch.uint8)
    return raw.view(-1)


def _inputs(case, seed):
    """The case's inputs, from the seed alone: raw weights, biases, activations."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, M = case["kind"], case["M"]
    d = {}
    if kind == "top":
        d["x"] = 3.0 * torch.randn(M, case["N"], generator=gen, device="cuda")
        return d
    if kind == "embedding":
        d["w"] = [_q8_0(gen, case["N"], case["K"])]
        d["ids"] = torch.randint(0, case["N"], (M,), generator=gen, device="cuda",
                                 dtype=torch.int32)
        return d
    d["x"] = torch.randn(M, case["K"], generator=gen, device="cuda")
    if kind == "matmul":
        d["w"] = [_q8_0(gen, case["K"], case["N"])]
        return d
    outs = _outputs(case)
    d["w"] = [_q8_0(gen, n, case["K"]) for n in outs]
    bias = case.get("bias", "none")
    dtype = {"none": None, "f32": torch.float32, "bf16": torch.bfloat16}[bias]
    d["bias"] = [None if dtype is None else
                 (0.1 * torch.randn(n, generator=gen, device="cuda")).to(dtype) for n in outs]
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    kind, M, K = case["kind"], case["M"], case.get("K")
    d["case"] = case

    def out(*shape, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device="cuda")

    if case.get("layout") == "tiled":  # the loader's re-tiling
        rows = _outputs(case)
        raw, d["w"] = d["w"], []
        for n, w in zip(rows, raw):
            t = torch.empty(capi.tiled_bytes(n, K), dtype=torch.uint8, device="cuda")
            capi.tile(w, t, n, K)
            d["w"].append(t)
    if kind == "top":
        k = min(case["k"], case["N"])
        d["ids"], d["probs"] = out(M, k, dtype=torch.int32), out(M, k)
    elif kind == "embedding":
        d["y"] = [out(M, K)]
    elif kind in ("matmul", "swiglu"):
        d["y"] = [out(M, case["N"])]
    else:
        d["y"] = [out(M, n) for n in _outputs(case)]
    if kind == "head":
        d["idx"], d["val"] = out(M, dtype=torch.int32), out(M)
    torch.cuda.synchronize()
    return d


def run(state):
    d, c = state, state["case"]
    kind, M, N, K = c["kind"], c["M"], c["N"], c.get("K")
    tiled = c.get("layout") == "tiled"
    if kind == "linear":
        if c["bias"] == "bf16":
            capi.linear_bias_bf16(d["x"], d["w"][0], d["bias"][0], d["y"][0], M, N, K,
                                  tiled=tiled)
        else:
            (capi.linear_tiled if tiled else capi.linear)(d["x"], d["w"][0], d["bias"][0],
                                                          d["y"][0], M, N, K)
        return d["y"]
    if kind == "multi":
        (capi.linear_multi_tiled if tiled else capi.linear_multi)(
            d["x"], d["w"], d["bias"], d["y"], _outputs(c), M, K)
        return d["y"]
    if kind == "swiglu":
        (capi.linear_swiglu_tiled if tiled else capi.linear_swiglu)(
            d["x"], d["w"][0], d["w"][1], d["y"][0], M, N, K)
        return d["y"]
    if kind == "head":
        (capi.linear_tiled if tiled else capi.linear)(d["x"], d["w"][0], None, d["y"][0], M, N,
                                                      K)
        capi.argmax(d["y"][0], M, N, d["idx"], d["val"])
        return [d["y"][0], d["idx"], d["val"]]
    if kind == "matmul":
        capi.matmul(d["x"], d["w"][0], d["y"][0], M, N, K)
        return d["y"]
    if kind == "embedding":
        (capi.embedding_tiled if tiled else capi.embedding)(d["w"][0], d["ids"], d["y"][0], M,
                                                            N, K)
        return d["y"]
    capi.top_tokens(d["x"], M, N, c["k"], d["ids"], d["probs"], temperature=c["temperature"])
    return [d["ids"], d["probs"]]


def work(case):
    kind, M, N, K = case["kind"], case["M"], case["N"], case.get("K")
    if kind == "top":
        return {"bytes": 4 * M * N + 8 * M * min(case["k"], N), "flops": 2 * M * N}
    if kind == "embedding":
        return {"bytes": M * (K // BLOCK) * BLOCK_BYTES + 4 * M + 4 * M * K, "flops": M * K}
    outs = _outputs(case)
    rows = sum(outs)
    written = N if kind == "swiglu" else rows
    width = {"none": 0, "f32": 4, "bf16": 2}[case.get("bias", "none")]
    n_bytes = rows * (K // BLOCK) * BLOCK_BYTES + 4 * M * K + 4 * M * written + width * rows
    if kind == "head":
        n_bytes += 8 * M
    return {"bytes": n_bytes, "flops": 2 * M * rows * K}


def tolerance(case):
    """Relative errors of the 2-norm against the exact result.

    fp32 sums (Linear and MatMul below 64 tokens): about 1e-7 with split sums, 1.3e-6 as
    one sequential fp32 chain of 4096 terms, which is as correct.  From 64 tokens on both
    operands are rounded once to bf16: 2.4e-3.  The gather is one exact product.  The
    head's index may move to another token only where two logits tie within rounding, and
    probabilities are fp32 sums of 152k exponentials."""
    kind = case["kind"]
    if kind == "embedding":
        return "exact"
    if kind == "top":
        return {"rel": 1e-5, "differ": 0.0}
    if kind == "head":
        return {"rel": 5e-6, "differ": 0.0}
    return {"rel": 1e-2 if case["M"] >= GEMM_TOKENS else 5e-6}


def exact(case, seed):
    d = _inputs(case, seed)
    kind, K = case["kind"], case.get("K")

    def dequant(raw, cols):
        b = raw.view(-1, BLOCK_BYTES)
        scale = b[:, :2].contiguous().view(torch.float16).double()
        return (b[:, 2:].contiguous().view(torch.int8).double() * scale).view(-1, cols)

    if kind == "embedding":
        return [dequant(d["w"][0], K)[d["ids"].long()]]
    x = d["x"].double()
    if kind == "top":
        k = min(case["k"], case["N"])
        # The scaled logits are fp32 values, as a sampler forms them.
        inv = torch.tensor(1.0, dtype=torch.float32) / torch.tensor(case["temperature"],
                                                                    dtype=torch.float32)
        scaled = (d["x"] * inv.item()).double()
        order = torch.sort(scaled, dim=1, descending=True, stable=True).indices[:, :k]
        return [order.to(torch.int32), torch.softmax(scaled, dim=1).gather(1, order)]
    if kind == "matmul":
        return [x @ dequant(d["w"][0], case["N"])]
    ys = [x @ dequant(w, K).t().contiguous() for w in d["w"]]
    ys = [y if b is None else y + b.double() for y, b in zip(ys, d["bias"])]
    if kind == "swiglu":
        return [ys[0] / (1.0 + torch.exp(-ys[0])) * ys[1]]
    if kind == "head":
        val, idx = ys[0].max(dim=1)
        return [ys[0], idx.to(torch.int32), val]
    return ys
