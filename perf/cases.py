"""The work that a user of this framework has it do, as cases with inputs, one pass, its useful work and its tolerance.

Three ways into the framework are covered: the attention operators on torch tensors (`ops.attn_fwd` / `ops.attn_bwd` as a
program with its own backward calls them, `ops.attention` and `ops.fused_attention` under torch autograd), from a single
head of 128 tokens to the 4096-token training shape, in both element types, with and without a band, with query heads
that share KV heads, at head sizes from 24 to 128; and `Llama`, whose training loop is the optimiser steps between two
saves followed by the parameters as numpy arrays.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from paperkiln_amd import ops
from paperkiln_amd.llama import Llama

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
LEARNING_RATE = 3e-4  # reached at the end of a pass: the linear warm-up a training run starts with


def _attention(name, B, T, Hq, Hkv, dk, dtype, api, causal=True, window=0, sinks=0, packed=False, std=1.0):
    """api: "direct" = attn_fwd + attn_bwd into buffers that the program keeps; "autograd" = attention() and a torch
    backward; "head" = fused_attention() on one head's [B*T, dk] matrix and a torch backward; "forward" = attn_fwd
    alone. packed: q, k and v are column slices of one fused projection, as a model's projection leaves them."""
    return {"name": name, "kind": "attention", "B": B, "T": T, "Hq": Hq, "Hkv": Hkv, "dk": dk, "dtype": dtype, "api": api,
            "causal": causal, "window": window, "sinks": sinks, "packed": packed, "std": std}


def _llama(name, vocab, d, layers, heads, d_ff, B, T, dtype, checkpoint, all_heads, steps, window=0, sinks=0):
    return {"name": name, "kind": "llama", "vocab": vocab, "d": d, "layers": layers, "heads": heads, "d_ff": d_ff, "B": B,
            "T": T, "dtype": dtype, "checkpoint": checkpoint, "all_heads": all_heads, "steps": steps, "window": window,
            "sinks": sinks}


def listed():
    return [
        # One head of the tiny Llama (d = 128, 4 heads, 4 stacked sequences of 128 tokens) through the reference's own
        # per-head operator: the smallest call there is, all launches and host time.
        _attention("head_fp32_tiny", 4, 128, 1, 1, 32, "fp32", "head"),
        # All heads of the fp32 parity configuration at once.
        _attention("fp32_small", 2, 128, 4, 4, 32, "fp32", "direct"),
        # A small story model's attention in training: short sequences, many of them.
        _attention("bf16_short", 16, 512, 8, 8, 64, "bf16", "autograd"),
        # Grouped-query attention of a half-billion-parameter model in training, 7 query heads to a KV head.
        _attention("bf16_gqa", 4, 2048, 14, 2, 64, "bf16", "autograd"),
        # Long-context training, full causal: the benchmark's headline shape.
        _attention("bf16_long", 4, 4096, 16, 16, 128, "bf16", "direct", std=0.5),
        # The same with a 256-token window and 4 sink tokens.
        _attention("bf16_window", 4, 4096, 16, 16, 128, "bf16", "direct", window=256, sinks=4, std=0.5),
        # Scoring one prompt of odd length with a large grouped-query model: forward only, heads read in the projection.
        _attention("bf16_prefill", 1, 3001, 32, 8, 128, "bf16", "forward", packed=True),
        # A bidirectional encoder in training on sequences of odd length, heads read in the projection.
        _attention("bf16_encoder", 6, 777, 12, 12, 64, "bf16", "autograd", causal=False, packed=True),
        # A head size between the usual ones.
        _attention("bf16_head80", 2, 1000, 8, 8, 80, "bf16", "autograd"),
        # Full-precision training, the reference's own element type, at an ordinary size.
        _attention("fp32_medium", 4, 1024, 8, 8, 64, "fp32", "direct"),
        # The tiny Llama trained in the reference's element type: 16 small steps, then a save.
        _llama("llama_tiny", 512, 128, 2, 4, 344, 4, 128, "fp32", False, True, 16),
        # The 35 M parameter Llama with activation checkpointing, bf16 over fp32 masters: 16 steps of 8192 tokens, a save.
        _llama("llama_35m", 32000, 512, 6, 8, 1376, 8, 1024, "bf16", True, False, 16),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_attention(rng):
    dtype = "bf16" if rng.random() < 0.7 else "fp32"
    u = rng.random()
    dk = 64 if u < 0.35 else 128 if u < 0.65 else 32 if u < 0.8 else rng.choice([24, 48, 80, 96])
    api = rng.choice(["direct", "autograd", "autograd", "forward", "head"])
    T = _log_uniform(rng, 48, 6000)
    tokens = min(16384, max(T, _log_uniform(rng, 128, 16384)))
    B = max(1, tokens // T)
    rep = rng.choice([1, 1, 1, 2, 4, 7])
    Hkv = rng.choice([1, 2, 4, 8, 16])
    if api == "head":
        rep = Hkv = 1
    while rep * Hkv > 1 and (rep * Hkv > 32 or rep * Hkv * dk > 4096 or B * T * rep * Hkv * dk > 4 * 4096 * 16 * 128):
        if Hkv > 1:
            Hkv //= 2
        else:
            rep = max(1, rep // 2)
    window = sinks = 0
    causal = True
    if api != "head":
        u = rng.random()
        if u < 0.2:
            causal = False
        elif u < 0.45:
            window, sinks = _log_uniform(rng, 16, max(17, T - 1)), rng.choice([0, 1, 4, 16])
    case = _attention("", B, T, rep * Hkv, Hkv, dk, dtype, api, causal, window, sinks, api != "head" and rng.random() < 0.5,
                      rng.choice([0.5, 1.0]))
    del case["name"]
    return case


def _draw_llama(rng):
    d = rng.choice([64, 128, 192, 256, 384, 512])
    heads = d // rng.choice([32, 64, 64])
    layers = rng.randint(1, 6)
    T = _log_uniform(rng, 32, 1024)
    B = max(1, _log_uniform(rng, 64, 8192) // T)
    dtype = "bf16" if rng.random() < 0.6 else "fp32"
    # full precision runs at a sixteenth of the matrix rate: users keep those models small
    vocab = _log_uniform(rng, 128, 32000 if dtype == "bf16" else 4000)
    window, sinks = (_log_uniform(rng, 16, max(17, T)), 4) if rng.random() < 0.2 else (0, 0)
    case = _llama("", vocab, d, layers, heads, (8 * d // 3 + 7) // 8 * 8, B, T, dtype, rng.random() < 0.5, rng.random() < 0.7,
                  rng.randint(8, 16), window, sinks)
    del case["name"]
    return case


def draw(rng):
    return _draw_llama(rng) if rng.random() < 0.25 else _draw_attention(rng)


def _prepare_attention(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)
    B, T, Hq, Hkv, dk, dtype = case["B"], case["T"], case["Hq"], case["Hkv"], case["dk"], DTYPES[case["dtype"]]

    def normal(*shape, std=1.0):
        return (torch.randn(shape, generator=gen, device=dev) * std).to(dtype)

    if case["api"] == "head":
        q, k, v = (normal(B * T, dk, std=case["std"]) for _ in range(3))
        d_o = normal(B * T, dk)
    elif case["packed"]:
        qkv = normal(B, T, Hq + 2 * Hkv, dk, std=case["std"])
        q, k, v = qkv[:, :, :Hq], qkv[:, :, Hq:Hq + Hkv], qkv[:, :, Hq + Hkv:]
        d_o = normal(B, T, Hq, dk)
    else:
        q = normal(B, T, Hq, dk, std=case["std"])
        k, v = (normal(B, T, Hkv, dk, std=case["std"]) for _ in range(2))
        d_o = normal(B, T, Hq, dk)
    state = {"case": case, "q": q, "k": k, "v": v, "d_o": d_o, "scale": float(np.float32(1.0 / math.sqrt(dk)))}
    if case["api"] in ("autograd", "head"):
        for name in ("q", "k", "v"):
            state[name] = state[name].detach().requires_grad_(True)
    elif case["api"] == "direct":  # gradients and scratch that a training loop keeps
        ws = ops.bwd_workspace_bytes(q, k, window=case["window"], sinks=case["sinks"])
        state["out"] = (torch.empty(q.shape, dtype=dtype, device=dev), torch.empty(k.shape, dtype=dtype, device=dev),
                        torch.empty(v.shape, dtype=dtype, device=dev), torch.empty(ws, dtype=torch.uint8, device=dev))
    return state


def _run_attention(s):
    c, q, k, v = s["case"], s["q"], s["k"], s["v"]
    if c["api"] == "head":
        o = ops.fused_attention(q, k, v, s["scale"], c["T"], c["causal"])
        dq, dk, dv = torch.autograd.grad(o, (q, k, v), s["d_o"])
        return {"o": o, "dq": dq, "dk": dk, "dv": dv}
    if c["api"] == "autograd":
        o = ops.attention(q, k, v, s["scale"], c["causal"], c["window"], c["sinks"])
        dq, dk, dv = torch.autograd.grad(o, (q, k, v), s["d_o"])
        return {"o": o, "dq": dq, "dk": dk, "dv": dv}
    o, lse = ops.attn_fwd(q, k, v, s["scale"], c["causal"], c["window"], c["sinks"])
    if c["api"] == "forward":
        return {"o": o, "lse": lse}
    dq, dk, dv = ops.attn_bwd(q, k, v, o, lse, s["d_o"], s["scale"], c["causal"], c["window"], c["sinks"], out=s["out"])
    return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}


def _prepare_llama(case, seed):
    model = Llama(case["vocab"], case["d"], case["layers"], case["heads"], case["d_ff"], compute_dtype=case["dtype"],
                  rope_all_heads=case["all_heads"], window=case["window"], sinks=case["sinks"], seed=seed % (1 << 31))
    n = case["B"] * case["T"]
    ids = np.random.RandomState(seed % (1 << 32)).randint(0, case["vocab"], (case["steps"], n + 1)).astype(np.int32)
    return {"case": case, "model": model, "batches": [(row[:-1].copy(), row[1:].copy()) for row in ids]}


def _run_llama(s):
    c, model = s["case"], s["model"]
    losses, norms = [], []
    for i, (x, y) in enumerate(s["batches"]):
        loss, _ = model.loss_backward(x, y, c["T"], checkpoint=c["checkpoint"])
        norms.append(model.adamw_step(LEARNING_RATE * (i + 1) / len(s["batches"]), max_norm=1.0))
        losses.append(loss)
    return {"losses": np.array(losses, np.float32), "norms": np.array(norms, np.float32), "params": model.params()}


def prepare(case, seed):
    return _prepare_llama(case, seed) if case["kind"] == "llama" else _prepare_attention(case, seed)


def run(state):
    return _run_llama(state) if state["case"]["kind"] == "llama" else _run_attention(state)


def _pairs(T, causal, window, sinks):
    """Visible (query, key) pairs of one head."""
    if not causal:
        return T * T
    if window <= 0 or window >= T:
        return T * (T + 1) // 2
    inside = window * (window + 1) // 2 + (T - window) * window
    first = T - window  # queries whose band starts past key 0: query i sees min(sinks, i + 1 - window) sink keys as well
    s = min(sinks, first)
    return inside + s * (s + 1) // 2 + (first - s) * s


def work(case):
    if case["kind"] == "llama":
        n, d, L = case["B"] * case["T"], case["d"], case["layers"]
        linear = L * (4 * d * d + 3 * d * case["d_ff"])
        params = linear + case["vocab"] * d + (2 * L + 1) * d
        attention = 14.0 * d * L * case["B"] * _pairs(case["T"], True, case["window"], case["sinks"])
        # every step: products forward and twice backward, tied head included; parameters and both moments in and out
        return {"flops": case["steps"] * (6.0 * n * (linear + case["vocab"] * d) + attention),
                "bytes": case["steps"] * 24.0 * params}
    B, T, Hq, Hkv, dk = (case[x] for x in ("B", "T", "Hq", "Hkv", "dk"))
    unit = 2.0 * dk * _pairs(T, case["causal"], case["window"], case["sinks"]) * B * Hq  # one product over the visible pairs
    es = 2 if case["dtype"] == "bf16" else 4
    q, kv, lse = B * T * Hq * dk * es, B * T * Hkv * dk * es, B * Hq * T * 4
    if case["api"] == "forward":
        return {"flops": 2 * unit, "bytes": 2.0 * q + 2 * kv + lse}
    return {"flops": 7 * unit, "bytes": 6.0 * q + 6 * kv + 2 * lse}


def tolerance(case):
    if case["kind"] == "llama":
        # The parameters after a pass are fp32 in both element types, moved by gradients of the compute type. AdamW divides
        # a gradient by the root of its second moment: where it is near zero its rounding decides an update's sign, so
        # single parameters may differ by a few updates while all of them together agree. Two GEMM libraries and two
        # forms of the head's loss differ by 8e-4 (largest 4e-2) in bf16; two orders of the head's sums by 6e-7 (1e-4) in fp32.
        return {"rel": 3e-3, "max": 0.2} if case["dtype"] == "bf16" else {"rel": 1e-5, "max": 1e-2}
    return {"rel": 1e-2, "max": 0.2} if case["dtype"] == "bf16" else {"rel": 1e-5, "max": 1e-3}
