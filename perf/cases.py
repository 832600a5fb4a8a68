"""Workloads that the speed of this library is judged by.

Each case is a call (or a step) of the public Python surface on tensors that are resident on the GPU, as a training
loop, an inference server or a script written for the reference would issue it.  ``listed`` holds one fixed size per
use, ``draw`` the ranges those sizes stand for.

Kinds of case:
  "serve"    ``Int8Linear`` without autograd on a module whose weight is quantised once: decode, prefill
  "train"    ``Int8Linear`` forward and backward through autograd, as a model calls it
  "step"     ``linear_fwd_bwd``: Y, dX and dW of one layer in one call
  "script"   ``fwd_32`` / ``bwd_33`` of a reference script's module: both bf16 operands quantised, then multiplied
  "decoder"  ``DecoderLayer`` forward and backward, its seven linears in int8
"""
import importlib
import math

import torch

import triton_int8_amd as T

__all__ = ["listed", "draw", "prepare", "run", "work", "tolerance"]

DEVICE = "cuda:0"
BF16 = torch.bfloat16


def _linear(kind, tokens, k, n, scheme="block_channel", hadamard="none", bias=False):
    return {"kind": kind, "tokens": tokens, "k": k, "n": n, "scheme": scheme, "hadamard": hadamard, "bias": bias}


def _script(api, half, batch, m, n, k):
    return {"kind": "script", "api": api, "half": half, "batch": batch, "m": m, "n": n, "k": k}


def _decoder(batch, seq, hidden, heads, mlp):
    return {"kind": "decoder", "batch": batch, "seq": seq, "hidden": hidden, "heads": heads, "mlp": mlp}


def listed():
    return [
        # one token of a single decode stream through a square projection: latency and launches are all there is
        {"name": "decode_1", **_linear("serve", 1, 4096, 4096)},
        # a decode batch through an MLP's up projection, per-row scales: streaming 56 MiB of int8 weight
        {"name": "decode_batch_37", **_linear("serve", 37, 4096, 14336, "double_channel")},
        # the prompt of one request, not a multiple of any tile, through an MLP's down projection with a bias
        {"name": "prefill_1000", **_linear("serve", 1000, 14336, 4096, bias=True)},
        # fine-tuning on very few tokens: every weight is quantised both ways for them
        {"name": "step_16", **_linear("step", 16, 4096, 4096)},
        # a module in a small training run: ragged token count, bias, mid-size model
        {"name": "train_1500_bias", **_linear("train", 1500, 2048, 5632, bias=True)},
        # a mid-size batch with per-token activation scales
        {"name": "step_row_block_3072", **_linear("step", 3072, 4096, 4096, "row_block")},
        # the headline layer of the benchmark: 8192 tokens, 4096 -> 4096, block-channel
        {"name": "step_8192", **_linear("step", 8192, 4096, 4096)},
        # the benchmark's gate / up projection with per-row scales on both operands
        {"name": "step_double_16384", **_linear("step", 16384, 4096, 14336, "double_channel")},
        # the same scheme with the rotation over the whole contraction dim in front of every quantiser
        {"name": "step_double_rotated_8192", **_linear("step", 8192, 4096, 4096, "double_channel", "full")},
        # the benchmark's heavy-tailed layer: 128-point rotation in front of every block quantiser
        {"name": "step_rotated_8192", **_linear("step", 8192, 8192, 8192, hadamard="128")},
        # the reference's own latency script at its shape, quantise-in-the-kernel arithmetic
        {"name": "script_fused_fwd", **_script("fused", "fwd", 4, 8192, 8192, 8192)},
        # a whole layer of a model in training at the benchmark's size
        {"name": "decoder_16384", **_decoder(4, 4096, 4096, 32, 14336)},
    ]


def _log_int(rng, lo, hi):
    """An integer between lo and hi, uniform over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng, lo, hi):
    """A feature count: a multiple of 128, odd multiples among them."""
    return 128 * max(lo // 128, min(hi // 128, _log_int(rng, lo, hi) // 128))


def draw(rng):
    kind = rng.choice(["serve", "serve", "train", "train", "step", "step", "step", "script", "decoder"])
    if kind == "decoder":
        heads = rng.choice([8, 16, 32])
        hidden = heads * rng.choice([64, 128])
        return _decoder(rng.randint(1, 4), 8 * _log_int(rng, 16, 512), hidden, heads, _features(rng, 2 * hidden, 7 * hidden // 2))
    if kind == "script":
        api = rng.choice(["block_channel", "double_channel", "fused", "tilelang"])
        half = rng.choice(["fwd", "bwd"])
        m, n = _features(rng, 256, 8192), _features(rng, 256, 8192)
        # the rotation of the double-channel scripts wants whole powers of two, the TileLang forward 256-wide groups
        k = 2 ** rng.randint(11, 13) if api == "double_channel" else 2 * _features(rng, 256, 4096)
        return _script(api, half, rng.randint(1, 4), m, n, k)
    scheme, hadamard = rng.choice([("block_channel", "none"), ("block_channel", "none"), ("double_channel", "none"),
                                   ("row_block", "none"), ("block_channel", "128"), ("row_block", "128"), ("double_channel", "full")])
    k, n = _features(rng, 1024, 14336), _features(rng, 1024, 14336)
    if hadamard == "full":
        k, n = 2 ** rng.randint(10, 13), 2 ** rng.randint(10, 13)
    if kind == "serve":
        tokens = _log_int(rng, 1, 8192)
    else:
        tokens = _log_int(rng, 16, 16384)
        if rng.random() < 0.3:                  # packed batches: whole tiles
            tokens = -(-tokens // 128) * 128
        if hadamard == "full":                  # the token dim is rotated too
            tokens = 2 ** max(7, min(14, int(math.log2(tokens))))
    return _linear(kind, tokens, k, n, scheme, hadamard, bias=kind != "step" and rng.random() < 0.4)


def _normal(gen, *shape, std=1.0):
    return (torch.randn(*shape, generator=gen, device=DEVICE, dtype=torch.float32) * std).to(BF16)


def _activations(gen, rows, cols, heavy_tailed=False):
    """N(0, 1) with 1 % of the channels x20, or Student-t with 3 degrees of freedom where a rotation is there to tame it."""
    x = torch.randn(rows, cols, generator=gen, device=DEVICE, dtype=torch.float32)
    if heavy_tailed:
        chi2 = sum(torch.randn(rows, cols, generator=gen, device=DEVICE, dtype=torch.float32).square_() for _ in range(3))
        x.div_(chi2.div_(3.0).sqrt_())
    else:
        x[:, torch.randperm(cols, generator=gen, device=DEVICE)[: -(-cols // 100)]] *= 20.0
    return x.to(BF16)


def _hadamard(case):
    return {"none": None, "128": 128, "full": "full"}[case["hadamard"]]


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    if kind == "script":
        module = importlib.import_module(f"triton_int8_amd.{_SCRIPTS[case['api']][case['half']]}")
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        a = _normal(gen, b, m, k)
        w = _normal(gen, n, k) if case["half"] == "fwd" else _normal(gen, b, n, k)
        return {"kind": kind, "call": module.fwd_32 if case["half"] == "fwd" else module.bwd_33, "a": a, "b": w}
    if kind == "decoder":
        layer = T.DecoderLayer(case["hidden"], case["heads"], case["mlp"], device=DEVICE)
        with torch.no_grad():
            for p in layer.parameters():
                p.copy_(_normal(gen, *p.shape, std=0.02) if p.dim() == 2 else 1.0 + _normal(gen, *p.shape, std=0.02))
        shape = (case["batch"], case["seq"], case["hidden"])
        x = _normal(gen, *shape).requires_grad_(True)
        return {"kind": kind, "layer": layer, "x": x, "dy": _normal(gen, *shape, std=1e-3), "wanted": [x, *layer.parameters()]}
    tokens, k, n = case["tokens"], case["k"], case["n"]
    x = _activations(gen, tokens, k, heavy_tailed=case["hadamard"] == "128")
    weight = _normal(gen, n, k, std=0.02)
    if kind == "step":
        return {"kind": kind, "x": x, "w": weight, "dy": _normal(gen, tokens, n, std=1e-3), "scheme": case["scheme"], "hadamard": _hadamard(case)}
    layer = T.Int8Linear(k, n, bias=case["bias"], scheme=case["scheme"], hadamard=_hadamard(case), device=DEVICE)
    with torch.no_grad():
        layer.weight.copy_(weight)
        if layer.bias is not None:
            layer.bias.copy_(_normal(gen, n))
        if kind == "serve":
            layer(x)                            # a server's first request quantises the weight
            return {"kind": kind, "layer": layer, "x": x}
    x.requires_grad_(True)
    return {"kind": kind, "layer": layer, "x": x, "dy": _normal(gen, tokens, n, std=1e-3), "wanted": [x, *layer.parameters()]}


_SCRIPTS = {
    "block_channel": {"fwd": "block_channel_fwd32", "bwd": "block_channel_bwd33"},
    "double_channel": {"fwd": "double_channel_fwd32", "bwd": "double_channel_bwd33"},
    "fused": {"fwd": "fused_fwd32", "bwd": "fused_bwd33"},
    "tilelang": {"fwd": "tilelang_block_channel_fwd", "bwd": "tilelang_block_channel_bwd"},
}


def run(state):
    kind = state["kind"]
    if kind == "script":
        return state["call"](state["a"], state["b"])
    if kind == "step":
        return T.linear_fwd_bwd(state["x"], state["w"], state["dy"], state["scheme"], state["hadamard"])
    if kind == "serve":
        with torch.no_grad():
            return state["layer"](state["x"])
    y = state["layer"](state["x"])
    return [y.detach(), *torch.autograd.grad(y, state["wanted"], state["dy"])]


def work(case):
    """bf16 inputs read once and outputs written once (a served weight: its int8 form), and the products' operations."""
    kind = case["kind"]
    if kind == "script":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        return {"bytes": 2 * (b * m * k + (1 if case["half"] == "fwd" else b) * n * k + b * m * n), "flops": 2 * b * m * n * k}
    if kind == "decoder":
        h, tokens = case["hidden"], case["batch"] * case["seq"]
        weights = 4 * h * h + 3 * h * case["mlp"]
        causal = 2 * case["batch"] * case["seq"] ** 2 * h            # half of Q K^T and of P V; the backward makes 2.5 times that
        return {"bytes": 2 * (2 * weights + 4 * tokens * h), "flops": int(6 * tokens * weights + 3.5 * causal)}
    tokens, k, n = case["tokens"], case["k"], case["n"]
    if kind == "serve":
        return {"bytes": n * k + 2 * tokens * (k + n), "flops": 2 * tokens * n * k}
    return {"bytes": 4 * (tokens * k + tokens * n + n * k), "flops": 6 * tokens * n * k}


def tolerance(case):
    if case["kind"] == "decoder":
        # int8 codes behind bf16 activations: the linears' products in 64 bits move single gradients by up to 2.8e-2 (and the
        # two RMSNorms without their rounding to bf16 in the middle by 4.7e-2), single elements by their own size
        return {"rel": 3e-2, "max": 0.99}
    double = case["scheme"] == "double_channel" if "scheme" in case else case["api"] == "double_channel"
    if double and not case.get("bias", False):
        return "exact"                          # int32 sums and a fixed order of roundings: one right answer
    # the products in 64 bits: up to 3.3e-5 away.  Those are bf16 outputs that round the other way, each by one ulp (at most
    # 2^-7 of the value); a bias rounds a second time, and what is left after it may be smaller than what was rounded before
    return {"rel": 1.2e-4, "max": 4e-2 if case.get("bias", False) else 2e-2}
