"""Upper bounds on activations, known at compile time.

An fp32 product runs on fp16 pairs (csrc/kh_gemm_f16.hip) only where its
activations have a bound that holds for every input of the graph: their fixed
power-of-two scale then never overflows fp16. In a pre-LN transformer every
product has one: a LayerNorm's output is at most sqrt(C) max|gamma| + max|beta|
whatever its input, a product with constant weights at most (row norm of its
input) * (largest column norm of the weights), attention's output at most the
largest |v|, and GELU, ReLU, tanh do not enlarge. A graph input has none.

Bounds are for finite values: a NaN stays a NaN in fp16, and no infinity
arises within a finite bound (a non-finite constant gives no bound).
"""

from __future__ import annotations

import math

import torch

from kiln.hip import lib as kl

NONE = (math.inf, math.inf)   # (largest magnitude, largest L2 norm of a row along the last dim)


def _up(x: float) -> float:
    """x rounded up to a power of two (so plans depend on constants' values
    through few distinct numbers)."""
    return x if x == 0.0 or not math.isfinite(x) else 2.0 ** math.ceil(math.log2(x))


class Bounds:
    """Bounds of a lowered graph's values. ``row_pattern(kernel)`` recognises a
    LayerNorm kernel: (1/C factor of the variance, gamma, beta) or None."""

    def __init__(self, graph, layer_norm, attention_value):
        self.g = graph
        self.layer_norm = layer_norm
        self.attention_value = attention_value
        self._known = {}
        self._norms = {}

    def largest(self, v) -> float:
        return self.of(v)[0]

    def of(self, v):
        if v not in self._known:
            self._known[v] = NONE   # (a cycle cannot occur; a missing rule means no bound)
            top, norm = self._of(v)
            norm = min(norm, top * math.sqrt(v.shape[-1] if v.type.rank else 1))
            top = min(top, norm)
            self._known[v] = (_up(top), _up(norm)) if math.isfinite(top) else NONE
        return self._known[v]

    def _constant(self, v):
        """The constant's values, or None when v is not one."""
        if v.node is None or v.node.op != "const":
            return None
        data = self.g.const_data(v)
        return None if data is None else torch.as_tensor(data, dtype=torch.float32)

    def _column_norm(self, b) -> float:
        """Largest L2 norm of a column (along K) of a [.., K, N] constant."""
        if b not in self._norms:
            node, perm = b.node, False
            if node is not None and node.op == "transpose" and b.type.rank == 2:
                node, perm = node.inputs[0].node, True
            data = self._constant(node.out) if node is not None else None
            self._norms[b] = float(torch.linalg.vector_norm(data, dim=-1 if perm else -2).max()) \
                if data is not None and data.dim() >= 2 and data.numel() else math.inf
        return self._norms[b]

    def _of(self, v):
        node = v.node
        if node is None:
            return NONE
        kernel = self.g.kernel_of(node)
        if kernel is not None and kernel.kind == "attention":
            value = self.attention_value(kernel, v)
            return (self.largest(value), math.inf) if value is not None else NONE
        if kernel is not None and kernel.kind == "reduction":
            found = self.layer_norm(kernel, v)
            if found is not None:
                c2, gamma, beta = found
                if not c2 > 0.0:
                    return NONE
                scale = 1.0 / math.sqrt(c2)   # |x - mean| / sqrt(c2 sum (x - mean)^2 + eps), and its row norm
                gt = self.of(gamma)[0] if gamma is not None else 1.0
                bt, bn = self.of(beta) if beta is not None else (0.0, 0.0)
                return gt * scale + bt, gt * scale + bn
        op, ins = node.op, node.inputs
        if op == "const":
            data = self._constant(v)
            if data is None or not data.numel() or not bool(torch.isfinite(data).all()):
                return NONE
            top = float(data.abs().max())
            return top, float(torch.linalg.vector_norm(data, dim=-1).max()) if data.dim() else top
        if op == "matmul":
            a_norm = self.of(ins[0])[1]
            return (a_norm * self._column_norm(ins[1]), math.inf) if math.isfinite(a_norm) else NONE
        if op in ("neg", "copy", "relu", "gelu"):   # |gelu(x)| <= |x|
            return self.of(ins[0])
        if op in ("tanh", "sigmoid", "erf"):
            return 1.0, math.inf
        if op in ("add", "sub"):
            (at, an), (bt, bn) = self.of(ins[0]), self.of(ins[1])
            whole = ins[0].shape[-1:] == v.shape[-1:] and ins[1].shape[-1:] == v.shape[-1:]
            return at + bt, an + bn if whole else math.inf
        if op in ("maximum", "minimum"):
            return max(self.largest(ins[0]), self.largest(ins[1])), math.inf
        if op == "mul":
            at, bt = self.largest(ins[0]), self.largest(ins[1])
            return (at * bt, math.inf) if math.isfinite(at) and math.isfinite(bt) else NONE
        if op in ("transpose", "reshape", "slice", "expand"):
            top, norm = self.of(ins[0])
            same_rows = op == "reshape" and ins[0].shape[-1:] == v.shape[-1:]
            return top, norm if same_rows else math.inf
        return NONE
