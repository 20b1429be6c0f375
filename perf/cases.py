"""Performance cases of the GEMM-family operators: what a program calls them with.

A case is a dict of plain values: ``op`` names the public entry point, the other keys its
sizes, types and layout.  ``listed()`` gives the fixed cases, ``draw(rng)`` one more of the
same ranges:

==============  ===========================================================================
``linear``      ``gemm`` / ``gemm_<bias>_<act>``: 1 to 8192 rows, N and K from 256 to 14336,
                bf16 / fp16 / fp32, weights as a ``W.t()`` view ("nk") or ``[K, N]`` ("kn"),
                sizes on and off the multiples of 64
``backward``    ``gemm_backward``: 64 to 8192 rows, N and K from 256 to 8192, bf16 / fp16
``batched``     ``batched_gemm``: 2 to 128 products of 64 to 2048 rows and columns, K from
                64 to 1024, bf16 / fp16
``blockscale``  ``gemm_a8w8_blockscale``: 1 to 8192 rows, N and K multiples of 128
``a8w8``        ``gemm_a8w8``: fp8 / int8, 1 to 8192 rows, any N and K
``moe``         ``fused_moe``: 1 to 8192 tokens, 8 to 64 experts, 1 to 8 per token
``grouped``     ``grouped_gemm`` / ``grouped_gemm_fp8``: 64 to 8192 tokens over 8 to 64
                unevenly loaded experts, any N and K
==============  ===========================================================================
"""

from __future__ import annotations

import math

import torch

import kore_amd
from kore_amd import workloads as W

_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}

# A drawn case costs at most what the largest listed one does (moe_prefill: 2.9 TFLOP).  The
# 32-bit, the two-way and the unaligned 8-bit products take longer for the same work.
_MAX_MNK = {"linear": 1 << 38, "fp32": 1 << 36, "backward": 1 << 37, "batched": 1 << 36,
            "blockscale": 1 << 38, "a8w8": 1 << 35, "moe": 1 << 37, "grouped": 1 << 36}


def listed():
    return [
        # one small layer for a few dozen rows: launch latency
        {"name": "linear_small", "op": "linear", "entry": "gemm", "dtype": "bf16", "layout": "kn",
         "M": 64, "N": 512, "K": 512},
        # a projection while 64 sequences decode: the weights are read once for few rows
        {"name": "linear_decode", "op": "linear", "entry": "gemm", "dtype": "bf16", "layout": "nk",
         "M": 64, "N": 4096, "K": 4096},
        # an MLP's first layer with its activation, and a reduction that ends off the tile
        {"name": "linear_act_ktail", "op": "linear", "entry": "gemm_bias_gelu", "dtype": "fp16", "layout": "kn",
         "M": 512, "N": 4096, "K": 4095},
        # a linear layer's backward in training: both gradients of 8192 tokens
        {"name": "backward_train", "op": "backward", "dtype": "bf16", "M": 8192, "N": 4096, "K": 4096},
        # a batch of medium products with an odd column count
        {"name": "batched_ragged", "op": "batched", "dtype": "bf16", "B": 8, "M": 512, "N": 513, "K": 512},
        # block-scaled fp8 weights while 128 sequences decode, and over a prompt
        {"name": "blockscale_decode", "op": "blockscale", "M": 128, "N": 7168, "K": 4096},
        {"name": "blockscale_prefill", "op": "blockscale", "M": 2048, "N": 7168, "K": 4096},
        # quantised decode where the reduction is not a multiple of the tile
        {"name": "a8w8_decode_ktail", "op": "a8w8", "kind": "int8", "mode": "pertoken",
         "M": 64, "N": 4096, "K": 4095},
        # mixture of experts: few tokens through large experts, a mid-size batch through many
        # small ones, a long prompt through large ones
        {"name": "moe_decode", "op": "moe", "T": 64, "E": 8, "topk": 2, "D": 4096, "I": 14336},
        {"name": "moe_mid", "op": "moe", "T": 512, "E": 32, "topk": 8, "D": 1024, "I": 768},
        {"name": "moe_prefill", "op": "moe", "T": 4096, "E": 8, "topk": 2, "D": 4096, "I": 14336},
        # one expert per token, unevenly loaded experts, fp8 weights
        {"name": "grouped_fp8", "op": "grouped", "kind": "fp8", "M": 4096, "E": 32, "N": 2048, "K": 4096},
    ]


# --------------------------------------------------------------------------- #
# Drawn cases
# --------------------------------------------------------------------------- #
def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _rows(rng, lo, hi):
    # token counts: any number, or a power of two
    m = _log(rng, lo, hi)
    return 1 << (m.bit_length() - 1) if rng.random() < 0.3 and (1 << (m.bit_length() - 1)) >= lo else m


def _dim(rng, lo, hi, step=64, ragged=0.3):
    # layer widths: mostly multiples of `step`, now and then any number
    d = _log(rng, lo, hi)
    return d if rng.random() < ragged else max(step, d // step * step)


def draw(rng):
    while True:
        case = _draw(rng)
        if _mnk(case) <= _MAX_MNK["fp32" if case.get("dtype") == "fp32" else case["op"]]:
            return case


def _mnk(c):
    if c["op"] == "moe":
        return 3 * c["T"] * c["topk"] * c["D"] * c["I"]
    return c.get("B", 1) * c["M"] * c["N"] * c["K"]


def _draw(rng):
    op = rng.choice(["linear", "linear", "linear", "backward", "batched", "blockscale", "a8w8", "a8w8",
                     "moe", "moe", "grouped"])
    if op == "linear":
        entry = rng.choice(["gemm"] * 4 + sorted(kore_amd.GEMM_FUSION_OPS))
        dtype = "bf16" if entry == "gemm" else rng.choice(["bf16", "fp16", "fp32"])
        return {"op": op, "entry": entry, "dtype": dtype, "layout": rng.choice(["nk", "kn"]),
                "M": _rows(rng, 1, 8192), "N": _dim(rng, 256, 14336), "K": _dim(rng, 256, 14336)}
    if op == "backward":
        return {"op": op, "dtype": rng.choice(["bf16", "bf16", "fp16"]), "M": _rows(rng, 64, 8192),
                "N": _dim(rng, 256, 8192), "K": _dim(rng, 256, 8192)}
    if op == "batched":
        return {"op": op, "dtype": rng.choice(["bf16", "bf16", "fp16"]), "B": _log(rng, 2, 128),
                "M": _dim(rng, 64, 2048), "N": _dim(rng, 64, 2048), "K": _dim(rng, 64, 1024)}
    if op == "blockscale":
        return {"op": op, "M": _rows(rng, 1, 8192), "N": _dim(rng, 512, 14336, 128, 0.0),
                "K": _dim(rng, 512, 8192, 128, 0.0)}
    if op == "a8w8":
        return {"op": op, "kind": rng.choice(["fp8", "int8"]), "mode": rng.choice(["pertoken", "pertensor"]),
                "M": _rows(rng, 1, 8192), "N": _dim(rng, 512, 14336, 128), "K": _dim(rng, 512, 8192, 128)}
    if op == "moe":
        E, topk, D, I = rng.choice([(8, 2, 4096, 14336), (32, 8, 1024, 768), (8, 2, 1024, 1408), None]) or (
            rng.choice([8, 16, 32, 64]), rng.choice([1, 2, 4, 8]), 128 * rng.randint(4, 32), 128 * rng.randint(4, 32))
        return {"op": op, "T": _rows(rng, 1, 8192), "E": E, "topk": topk, "D": D, "I": I}
    return {"op": op, "kind": rng.choice(["bf16", "fp8"]), "M": _rows(rng, 64, 8192), "E": rng.choice([8, 16, 32, 64]),
            "N": _dim(rng, 512, 4096, 128, 0.2), "K": _dim(rng, 512, 4096, 128, 0.2)}


# --------------------------------------------------------------------------- #
# Inputs, one pass
# --------------------------------------------------------------------------- #
def prepare(case, seed):
    dev = torch.device("cuda")
    op = case["op"]
    if op == "linear":
        M, N, K, dtype = case["M"], case["N"], case["K"], _DT[case["dtype"]]
        has_bias = case["entry"].startswith("gemm_bias")
        a, b, bias = W.fused_inputs(M, N, K, seed=seed, device=dev, dtype=dtype, with_bias=has_bias)
        if case["layout"] == "kn":
            b = b.contiguous()
        return getattr(kore_amd, case["entry"]), ((a, b, bias) if has_bias else (a, b))
    if op == "backward":
        return kore_amd.gemm_backward, W.backward_inputs(case["M"], case["N"], case["K"], seed=seed, device=dev,
                                                         dtype=_DT[case["dtype"]])
    if op == "batched":
        B, M, N, K, dtype = case["B"], case["M"], case["N"], case["K"], _DT[case["dtype"]]
        g = torch.Generator(device=dev).manual_seed(seed)
        a = (torch.randn((B, M, K), generator=g, device=dev) / K ** 0.5).to(dtype)
        b = (torch.randn((B, N, K), generator=g, device=dev) / K ** 0.5).to(dtype)
        return kore_amd.batched_gemm, (a, b)
    if op == "blockscale":
        return kore_amd.gemm_a8w8_blockscale, W.fp8_inputs(case["M"], case["N"], case["K"], seed=seed, device=dev)
    if op == "a8w8":
        return kore_amd.gemm_a8w8, W.a8w8_inputs(case["M"], case["N"], case["K"], case["kind"], case["mode"],
                                                 seed=seed, device=dev)
    if op == "moe":
        return kore_amd.fused_moe, W.moe_inputs(case["T"], case["E"], case["topk"], case["D"], case["I"], seed=seed,
                                                device=dev)
    make, entry = ((W.grouped_fp8_inputs, kore_amd.grouped_gemm_fp8) if case["kind"] == "fp8"
                   else (W.grouped_inputs, kore_amd.grouped_gemm))
    return entry, make(case["M"], case["E"], case["N"], case["K"], seed=seed, device=dev,
                       router_bias=W.jagged_bias(case["E"]))


def run(state):
    entry, args = state
    return entry(*args)


# --------------------------------------------------------------------------- #
# What a pass cannot do without
# --------------------------------------------------------------------------- #
def _experts_used(rows, picks, probs):
    # experts that at least one of `rows` tokens picks, on average
    return sum(1.0 - (1.0 - min(1.0, picks * p)) ** rows for p in probs)


def work(case):
    op = case["op"]
    if op == "moe":
        T, E, topk, D, I = (case[k] for k in ("T", "E", "topk", "D", "I"))
        used = _experts_used(T, topk, [1.0 / E] * E)
        return {"bytes": used * 3 * D * I * 2 + T * D * 4 + T * topk * 8, "flops": 6 * T * topk * D * I}
    M, N, K, B = case["M"], case["N"], case["K"], case.get("B", 1)
    if op == "linear":
        es = _SIZE[case["dtype"]]
        bias = N if case["entry"].startswith("gemm_bias") else 0
        return {"bytes": (M * K + N * K + M * N + bias) * es, "flops": 2 * M * N * K}
    if op == "backward":
        return {"bytes": 2 * (M * K + N * K) * 2 + M * N * 2, "flops": 4 * M * N * K}
    if op == "batched":
        return {"bytes": B * (M * K + N * K + M * N) * 2, "flops": 2 * B * M * N * K}
    if op == "blockscale":
        return {"bytes": M * K + N * K + 2 * M * N + (M * K // 128 + N * K // 128 ** 2) * 4, "flops": 2 * M * N * K}
    if op == "a8w8":
        return {"bytes": M * K + N * K + 2 * M * N + 4 * (M + N), "flops": 2 * M * N * K}
    weights = torch.softmax(W.jagged_bias(case["E"]).double(), 0).tolist()
    used = _experts_used(M, 1, weights)
    es = 1 if case["kind"] == "fp8" else 2
    scales = 4 * (M + used * N) if case["kind"] == "fp8" else 0
    return {"bytes": (M * K + used * N * K) * es + 2 * M * N + 4 * M + scales, "flops": 2 * M * N * K}


# --------------------------------------------------------------------------- #
# How exact the results are
# --------------------------------------------------------------------------- #
def tolerance(case):
    # Sums are held in 32 bits and rounded once to the result's type, so two correct
    # implementations differ where a sum falls on the other side of a rounding step.
    # Against 64 bits the relative error (2-norm), measured on the listed cases and fifty
    # drawn ones, is at most 1.8e-3 for bf16, 2.2e-4 for fp16 and 2.0e-6 for fp32 (a sum of
    # 11840 products); the bounds are about four times that.
    dtype = case.get("dtype", "bf16")
    return {"rel": {"bf16": 7e-3, "fp16": 9e-4, "fp32": 8e-6}[dtype]}


def _act64(x, entry):
    act = entry.rsplit("_", 1)[-1]
    if act == "relu":
        return x.clamp(min=0)
    if act == "gelu":
        return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))
    if act == "silu":
        return x * torch.sigmoid(x)
    if act == "tanh":
        return torch.tanh(x)
    if act == "sigmoid":
        return torch.sigmoid(x)
    return x


def exact(case, seed):
    _, args = prepare(case, seed)
    op = case["op"]
    if op == "linear":
        y = args[0].double() @ args[1].double()
        if len(args) == 3:
            y = y + args[2].double()
        return _act64(y, case["entry"])
    if op == "backward":
        x, w, dy = (t.double() for t in args)
        return dy @ w, dy.t().contiguous() @ x
    if op == "batched":
        a, b = args
        return torch.stack([a[i].double() @ b[i].double().t().contiguous() for i in range(a.shape[0])])
    if op == "blockscale":
        xq, wq, xs, ws = args
        x = xq.double() * xs.double().repeat_interleave(128, 1)
        w = wq.double() * ws.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
        return x @ w.t().contiguous()
    if op == "a8w8":
        xq, wq, xs, ws = args
        return (xq.double() @ wq.double().t().contiguous()) * xs.double() * ws.double()
    if op == "moe":
        hidden, w1, w2, tw, ti = args
        x = hidden.double()
        out = torch.zeros_like(x)
        for e in range(w1.shape[0]):
            t, k = torch.nonzero(ti == e, as_tuple=True)
            if t.numel() == 0:
                continue
            gate, up = (x[t] @ w1[e].double().t().contiguous()).chunk(2, dim=1)
            y = (gate * torch.sigmoid(gate) * up) @ w2[e].double().t().contiguous()
            out.index_add_(0, t, y * tw[t, k].double()[:, None])
        return out
    x, w, ids = args[0].double(), args[1], args[-1].long()
    if case["kind"] == "fp8":
        x = x * args[2].double()
    out = torch.zeros((x.shape[0], w.shape[1]), dtype=torch.float64, device=x.device)
    for e in ids.unique().tolist():
        we = w[e].double()
        if case["kind"] == "fp8":
            we = we * args[3][e].double()
        rows = ids == e
        out[rows] = x[rows] @ we.t().contiguous()
    return out
