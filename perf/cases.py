"""What a user of the framework runs, as cases whose speed can be measured.

Every case compiles a model with ``kiln.compile(..., device="cuda")`` and calls
the result, which is how a program uses the framework. A case is a dict:

  kind         what is compiled (see ``build``)
  tokens       rows of the activation (sequence length)
  d, heads     model width and attention heads, where the kind has them
  out          output width of a single Linear
  layers       number of blocks of a stack
  causal       whether attention has the upper-triangular -inf mask
  precision    "fp32" (the default), "tf32" (``allow_tf32=True``) or "bf16"
               (``matmul_precision="bf16"``)
  autotune     the compile flag of that name

The listed sizes are the GPT-2-small shapes of the benchmark configurations
(d 768, 12 heads of 64, MLP 3072) and odd ones in between; ``draw`` spreads
over the same ranges.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn as nn
import torch.nn.functional as F

# the package of the repository that is the working folder
sys.path.insert(0, os.path.abspath("kiln-compiler_amd"))

import kiln  # noqa: E402

INIT_STD = 0.02     # Linear weights and biases of the benchmark configurations


# -- the models a user brings ---------------------------------------------------------------


class LinearGelu(nn.Module):
    def __init__(self, d, out):
        super().__init__()
        self.fc = nn.Linear(d, out)

    def forward(self, x):
        return F.gelu(self.fc(x))


class Mlp(nn.Module):
    """The MLP half of a pre-LN block."""

    def __init__(self, d):
        super().__init__()
        self.ln = nn.LayerNorm(d)
        self.fc = nn.Linear(d, 4 * d)
        self.proj = nn.Linear(4 * d, d)

    def forward(self, x):
        return x + self.proj(F.gelu(self.fc(self.ln(x)), approximate="tanh"))


class Attention(nn.Module):
    """The attention half of a pre-LN block: causal, or over the whole sequence."""

    def __init__(self, d, heads, tokens, causal):
        super().__init__()
        self.heads = heads
        self.causal = causal
        self.ln = nn.LayerNorm(d)
        self.c_attn = nn.Linear(d, 3 * d)
        self.c_proj = nn.Linear(d, d)
        if causal:
            self.register_buffer("mask", torch.full((tokens, tokens), float("-inf")).triu(1))

    def forward(self, x):
        t, c = x.shape
        dh = c // self.heads
        q, k, v = (y.view(t, self.heads, dh).transpose(0, 1) for y in self.c_attn(self.ln(x)).split(c, dim=1))
        att = (q @ k.transpose(-2, -1)) * (1.0 / math.sqrt(dh))
        if self.causal:
            att = att + self.mask
        y = F.softmax(att, dim=-1) @ v
        return x + self.c_proj(y.transpose(0, 1).contiguous().view(t, c))


class Block(nn.Module):
    """GPT-2 block: causal attention, then the MLP, each with its residual."""

    def __init__(self, d, heads, tokens):
        super().__init__()
        self.attn = Attention(d, heads, tokens, True)
        self.mlp = Mlp(d)

    def forward(self, x):
        return self.mlp(self.attn(x))


class Stack(nn.Module):
    """`layers` blocks and the final LayerNorm (GPT-2 without its embeddings and head)."""

    def __init__(self, layers, d, heads, tokens):
        super().__init__()
        self.blocks = nn.ModuleList(Block(d, heads, tokens) for _ in range(layers))
        self.ln_f = nn.LayerNorm(d)

    def forward(self, x):
        for block in self.blocks:
            x = block(x)
        return self.ln_f(x)


class BiasGelu(nn.Module):
    def __init__(self, d):
        super().__init__()
        self.bias = nn.Parameter(torch.zeros(d))

    def forward(self, x):
        return F.gelu(x + self.bias, approximate="tanh")


class ScaledSoftmax(nn.Module):
    def forward(self, x):
        return F.softmax(x * 0.125, dim=-1)


def build(case, seed):
    """(model, input) on the CPU, from the seed alone."""
    kind, tokens, d = case["kind"], case["tokens"], case.get("d")
    if kind == "linear_gelu":
        model = LinearGelu(d, case["out"])
    elif kind == "mlp":
        model = Mlp(d)
    elif kind == "attention":
        model = Attention(d, case["heads"], tokens, case["causal"])
    elif kind == "block":
        model = Block(d, case["heads"], tokens)
    elif kind == "stack":
        model = Stack(case["layers"], d, case["heads"], tokens)
    elif kind == "bias_gelu":
        model = BiasGelu(d)
    else:
        model = ScaledSoftmax()
    gen = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for m in model.modules():
            if isinstance(m, nn.Linear):
                m.weight.normal_(0.0, INIT_STD, generator=gen)
                m.bias.normal_(0.0, INIT_STD, generator=gen)
            elif isinstance(m, nn.LayerNorm):
                m.weight.normal_(1.0, INIT_STD, generator=gen)
                m.bias.normal_(0.0, INIT_STD, generator=gen)
            elif isinstance(m, BiasGelu):
                m.bias.normal_(0.0, 1.0, generator=gen)
    shape = (case["heads"], tokens, tokens) if kind == "softmax" else (tokens, d)
    return model.eval(), torch.randn(*shape, generator=gen)


# -- the cases --------------------------------------------------------------------------------


def _case(name, kind, tokens, precision="fp32", autotune=False, **sizes):
    return {"name": name, "kind": kind, "tokens": tokens, **sizes, "precision": precision, "autotune": autotune}


def listed():
    return [
        # one Linear with its activation at a short prompt: a single launch
        _case("linear_gelu_128", "linear_gelu", 128, d=768, out=3072),
        # the memory-bound fused chains, as a model's own pieces
        _case("bias_gelu_2048x3072", "bias_gelu", 2048, d=3072),
        _case("softmax_12x512x512", "softmax", 512, heads=12),
        # half blocks at lengths that fit no tile, compiled with the defaults
        _case("mlp_333", "mlp", 333, d=768),
        _case("attention_full_600", "attention", 600, d=512, heads=8, causal=False),
        # the GPT-2 block: a short prompt, an odd length, the longest context
        _case("block_128", "block", 128, d=768, heads=12, autotune=True),
        _case("block_777", "block", 777, d=768, heads=12),
        _case("block_2048", "block", 2048, d=768, heads=12, autotune=True),
        # the reduced-precision options of the same block
        _case("block_tf32_1024", "block", 1024, "tf32", True, d=768, heads=12),
        _case("block_bf16_1024", "block", 1024, "bf16", True, d=768, heads=12),
        # whole calls: prefill of the 12-layer stack, and one token through it
        _case("stack12_prefill_1024", "stack", 1024, d=768, heads=12, layers=12, autotune=True),
        _case("stack12_decode", "stack", 1, d=768, heads=12, layers=12, autotune=True),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["linear_gelu", "mlp", "attention", "block", "block", "stack", "bias_gelu", "softmax"])
    precision = rng.choice(["fp32", "fp32", "fp32", "tf32", "bf16"])
    tokens = _log_int(rng, 8, 2048)
    heads, head = rng.choice([4, 6, 8, 12, 16]), rng.choice([32, 64, 64])
    d = heads * head
    if kind == "linear_gelu":
        sizes = {"d": _log_int(rng, 64, 3072), "out": _log_int(rng, 64, 3072)}
    elif kind == "mlp":
        sizes = {"d": d}
    elif kind == "attention":
        sizes = {"d": d, "heads": heads, "causal": rng.random() < 0.5}
    elif kind == "block":
        sizes = {"d": d, "heads": heads}
    elif kind == "stack":
        tokens = rng.choice([1, 1, _log_int(rng, 8, 512)])
        sizes = {"d": d, "heads": heads, "layers": rng.randint(2, 4)}
    elif kind == "bias_gelu":
        precision, sizes = "fp32", {"d": _log_int(rng, 64, 4096)}
    else:
        precision, tokens, sizes = "fp32", _log_int(rng, 8, 1024), {"heads": heads}
    return {"kind": kind, "tokens": tokens, **sizes, "precision": precision, "autotune": False}


# -- one pass ----------------------------------------------------------------------------------


def prepare(case, seed):
    model, x = build(case, seed)
    flags = {"allow_tf32": True} if case["precision"] == "tf32" else {"matmul_precision": case["precision"]}
    compiled = kiln.compile(model, (x,), device="cuda", autotune=case["autotune"], **flags)
    return {"compiled": compiled, "x": x.to("cuda")}


def run(state):
    return state["compiled"](state["x"])


def work(case):
    """Each input, weight and output once; a causal layer's visible pairs only."""
    kind, t, d = case["kind"], case["tokens"], case.get("d")
    weight = 2 if case["precision"] == "bf16" else 4
    if kind == "linear_gelu":
        n = case["out"]
        return {"bytes": 4 * t * (d + n) + weight * d * n, "flops": 2 * t * d * n}
    if kind == "bias_gelu":
        return {"bytes": 8 * t * d, "flops": 10 * t * d}
    if kind == "softmax":
        cells = case["heads"] * t * t
        return {"bytes": 8 * cells, "flops": 5 * cells}
    layers = case.get("layers", 1)
    pairs = t * (t + 1) // 2 if case.get("causal", True) else t * t
    attention = {"weights": 4 * d * d, "flops": 8 * t * d * d + 4 * pairs * d}
    mlp = {"weights": 8 * d * d, "flops": 16 * t * d * d}
    parts = {"mlp": [mlp], "attention": [attention]}.get(kind, [attention, mlp] * layers)
    return {"bytes": 8 * t * d + weight * sum(p["weights"] for p in parts), "flops": sum(p["flops"] for p in parts)}


def tolerance(case):
    """About four times the measured distance from ``exact``: 6e-8 for the
    fused chains, up to 4e-7 for fp32 blocks and 7.5e-7 for the 12 layers,
    4.5e-6 for three-pass bf16, 2.4e-3 for bf16 inputs."""
    if case["kind"] in ("bias_gelu", "softmax"):
        return {"rel": 5e-7}
    if case["precision"] == "bf16":
        return {"rel": 1e-2}
    if case["precision"] == "tf32":
        return {"rel": 2e-5}
    return {"rel": 4e-6 if case["kind"] == "stack" else 2e-6}


def exact(case, seed):
    model, x = build(case, seed)
    device = "cuda" if torch.cuda.is_available() else "cpu"
    with torch.no_grad():
        return model.double().to(device)(x.double().to(device))
