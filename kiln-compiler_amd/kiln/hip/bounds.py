"""How large activations can be, and how large they usually are.

An fp32 product runs on fp16 pairs (csrc/kh_gemm_f16.hip) with one fixed power
of two for all its activations, chosen at compile time. Two things are asked
of it, both answered here from the graph and its constants:

  * Safe: no value overflows fp16, whatever the input. That needs an upper
    bound. In a pre-LN transformer every product has one: a LayerNorm's output
    is at most sqrt(C) max|gamma| + max|beta| whatever its input, a product
    with constant weights at most (row norm of its input) * (largest column
    norm of the weights), attention's output at most the largest |v|, and GELU,
    ReLU, tanh do not enlarge. A graph input has none.

  * Tight: the values lie close enough under that bound. A pair holds 23 bits
    of a value near the bound but has an absolute floor (TIGHT below), and a
    bound grows by sqrt(N) per product that no LayerNorm follows, or with one
    outlier gain, where the values do not. So beside the bound goes each
    element's usual size: |gamma|, |beta| behind a LayerNorm (whose rows have
    norm sqrt(C)), root sums of squares through products and additions, half
    behind GELU and ReLU, a mean of `keys` independent values behind
    attention. A product takes pairs only where, for every output column, the
    bound is within TIGHT of the root mean square of what the column sums;
    elsewhere it stays on the fp32 matrix cores. A size is only claimed where
    it follows from the graph (an unknown one refuses). Cancellation needs no
    care: what cancels has been rounded in fp32 before, relative to the terms.

Bounds are for finite values: a NaN stays a NaN in fp16, and no infinity
arises within a finite bound (a non-finite constant gives no bound).
"""

from __future__ import annotations

import math
from dataclasses import dataclass

import torch

from kiln.hip import f16

NONE = (math.inf, math.inf)   # (largest magnitude, largest L2 norm of a row along the last dim)

# How far a bound may lie above the usual size. Below its 23 bits a pair adds,
# to a weight, at most 2^-39 of its column's largest, to q or k in a score
# 2^-39 of their bounds, to any other activation 2^-50 of its bound
# (csrc/kh_common.hpp); fp32 operands of the usual size bring 2^-25 of it each.
# At 2^13 the first two stay under half of that, and the third under 2^-12: a
# row may be 2^11 times smaller than usual (a LayerNorm's, where its spread is
# small against sqrt(eps)) before it is held less well. GPT-2 blocks of 2048
# tokens reach 2^10.4 (their output projection, behind attention) and 2^5
# elsewhere, where rows may be 2^19 times smaller.
TIGHT = 2.0 ** 13


@dataclass
class _Product:
    """A product with a constant: largest column norm of the weights, the
    output's size, and whether fp16 pairs hold both operands."""

    column_norm: float
    size: torch.Tensor
    tight: bool


class Bounds:
    """Bounds and sizes of a lowered graph's values. ``layer_norm(kernel, v)``
    recognises a LayerNorm kernel: (1/C factor of the variance, eps, gamma,
    beta) or None; ``attention(kernel)`` the match of an attention kernel."""

    def __init__(self, graph, layer_norm, attention):
        self.g = graph
        self.layer_norm = layer_norm
        self.attention = attention
        self._known = {}
        self._sizes = {}
        self._products = {}

    # -- what the lowering asks ------------------------------------------------------

    def pair_product(self, mm):
        """Exponent of the scale of matmul node mm's A operand if the product
        can run on fp16 pairs (safe and tight), else None."""
        e = f16.activation_exponent(self.largest(mm.inputs[0]))
        if e is None:
            return None
        return e if self.product(mm).tight else None

    def pair_attention(self, m):
        """Exponents of the scales of q, k and v of attention match m if it can
        run on fp16 pairs, else None. Scores are asked per head, as a dot
        product's operands are; v per head and dimension."""
        tops = [self.largest(v) for v in (m.q, m.k, m.v)]
        exponents = tuple(f16.activation_exponent(top) for top in tops)
        if None in exponents:
            return None
        q, k, v = (self.size(x) for x in (m.q, m.k, m.v))
        if m.k_transposed:
            k = k.transpose(-2, -1)
        # (a row's usual size: the smallest where it differs over the tokens)
        q, k, v = (x.amin(dim=-2) for x in (q, k, v))
        dh = m.q.shape[-1]
        q, k = (x.expand(*x.shape[:-1], dh) for x in (q, k))
        usual = TIGHT * (q * k).norm(dim=-1)
        ok = (tops[0] * k.norm(dim=-1) <= usual).all() and (tops[1] * q.norm(dim=-1) <= usual).all()
        return exponents if bool(ok) and bool((tops[2] <= TIGHT * v).all()) else None

    # -- upper bounds ----------------------------------------------------------------

    def largest(self, v) -> float:
        return self.of(v)[0]

    def of(self, v):
        if v not in self._known:
            self._known[v] = NONE   # (a cycle cannot occur; a missing rule means no bound)
            top, norm = self._of(v)
            norm = min(norm, top * math.sqrt(v.shape[-1] if v.type.rank else 1))
            top = min(top, norm)
            self._known[v] = (top, norm) if math.isfinite(top) else NONE
        return self._known[v]

    def _constant(self, v):
        """The constant's values, or None when v is not one."""
        if v.node is None or v.node.op != "const":
            return None
        data = self.g.const_data(v)
        return None if data is None else torch.as_tensor(data, dtype=torch.float32)

    def _norm_of(self, v):
        """(1/C factor, eps, gamma, beta) if v is a LayerNorm kernel's output."""
        kernel = self.g.kernel_of(v.node)
        return self.layer_norm(kernel, v) if kernel is not None and kernel.kind == "reduction" else None

    def _attention_of(self, node):
        """The match of the attention whose second product `node` is, else None."""
        kernel = self.g.kernel_of(node)
        if kernel is None or kernel.kind != "attention" or [n for n in kernel.nodes if n.op == "matmul"][-1] is not node:
            return None
        m = self.attention(kernel)
        return m if m is not None and node.inputs[1] is m.v else None

    def _of(self, v):
        node = v.node
        if node is None:
            return NONE
        found = self._norm_of(v)
        if found is not None:
            c2, eps, gamma, beta = found
            if not (c2 > 0.0 and eps >= 0.0):
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
            rows = data.double()
            return top, float(torch.linalg.vector_norm(rows, dim=-1).max()) if data.dim() else top
        if op == "matmul":
            m = self._attention_of(node)
            if m is not None:   # a weighted mean of rows of v
                return self.largest(m.v), math.inf
            a_norm = self.of(ins[0])[1]
            return (a_norm * self.product(node).column_norm, math.inf) if math.isfinite(a_norm) else NONE
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

    # -- usual sizes -----------------------------------------------------------------

    def size(self, v) -> torch.Tensor:
        """Usual magnitude of v's elements (float64, v's rank; a dim of 1 means
        alike along it); NaN where none is claimed."""
        if v not in self._sizes:
            unknown = _unknown(v.type.rank)
            self._sizes[v] = unknown
            found = self._size(v)
            self._sizes[v] = unknown if found is None or not bool(torch.isfinite(found).all()) else found
        return self._sizes[v]

    def _size(self, v):
        node = v.node
        if node is None:
            return None
        found = self._norm_of(v)
        if found is not None:
            _, _, gamma, beta = found
            shape = [1] * (v.type.rank - 1) + [v.shape[-1]]
            parts = [p.reshape(shape) if p.numel() == v.shape[-1] else p.amin()
                     for p in (self.size(x) for x in (gamma, beta) if x is not None)]
            gain = parts[0] if gamma is not None else torch.ones(shape, dtype=torch.float64)
            return torch.hypot(gain, parts[-1]) if beta is not None else gain
        op, ins = node.op, node.inputs
        if op == "const":
            data = self._constant(v)
            return None if data is None else data.double().abs()
        if op == "matmul":
            m = self._attention_of(node)
            if m is not None:
                return self.size(m.v).amin(dim=-2, keepdim=True) / math.sqrt(m.v.shape[-2])
            return self.product(node).size
        if op in ("neg", "copy"):
            return self.size(ins[0])
        if op in ("relu", "gelu"):
            return self.size(ins[0]) / 2
        if op in ("tanh", "erf"):
            s = self.size(ins[0])
            return s / torch.hypot(s, torch.ones_like(s))
        if op in ("add", "sub"):
            return torch.hypot(self.size(ins[0]), self.size(ins[1]))
        if op == "mul" and any(self._constant(x) is not None for x in ins):
            return self.size(ins[0]) * self.size(ins[1])
        if op == "transpose":
            return self.size(ins[0]).permute(node.attrs["perm"])
        if op == "expand":
            s = self.size(ins[0])
            return s.reshape([1] * (v.type.rank - s.dim()) + list(s.shape))
        if op == "slice":
            s, dim = self.size(ins[0]), node.attrs["dim"] % v.type.rank
            if s.shape[dim] == 1:
                return s
            index = torch.arange(node.attrs["start"], node.attrs["end"], node.attrs.get("step", 1))
            return s.index_select(dim, index) if index.numel() == v.shape[dim] else None
        if op == "reshape":
            return _reshaped(self.size(ins[0]), ins[0].shape, v.shape)
        return None

    # -- products with constants -----------------------------------------------------

    def product(self, mm) -> _Product:
        if mm not in self._products:
            self._products[mm] = self._product(mm)
        return self._products[mm]

    def _product(self, mm) -> _Product:
        a, b = mm.inputs
        rank = mm.out.type.rank
        none = _Product(math.inf, _unknown(rank), False)
        node, perm = b.node, False
        if node is not None and node.op == "transpose" and b.type.rank == 2:
            node, perm = node.inputs[0].node, True
        w = self._constant(node.out) if node is not None else None
        if w is None or w.dim() < 2 or not w.numel():
            return none
        w = w.transpose(-2, -1) if perm else w   # [.., K, N]
        # root sums of squares of the columns, plain and weighted by A's sizes,
        # from one pass over the squares; columns whose squares could overflow
        # or vanish are scaled by their largest weight first
        top = torch.maximum(w.amax(dim=-2), -w.amin(dim=-2)).double()
        if not bool(torch.isfinite(top).all()):
            return none
        unit = torch.where((top > 0) & ((top < 1e-12) | (top > 1e12)), top, torch.ones_like(top))
        scaled = bool((unit != 1).any())
        # the smallest size along the other dims, for every K
        s = self.size(a)
        while s.dim() > 1:
            s = s.amin(dim=0)
        s = s.expand(w.shape[-2])
        s_top = float(s.max()) or 1.0
        squares = (w / unit.float().unsqueeze(-2)).square_() if scaled else w.square()
        weighted = torch.stack([torch.ones_like(s), (s / s_top).square()]).float() @ squares   # [.., 2, N]
        norm = unit * weighted[..., 0, :].double().sqrt()
        usual = unit * s_top * weighted[..., 1, :].double().sqrt()
        tight = (bool((self.largest(a) * norm <= TIGHT * usual).all())
                 and bool((top * float(s.norm()) <= TIGHT * usual).all()) and f16.columns_fit(top))
        size = usual.unsqueeze(-2) if usual.dim() > 1 else usual
        return _Product(float(norm.max()), size.reshape([1] * (rank - size.dim()) + list(size.shape)), tight)


def _unknown(rank):
    return torch.full([1] * rank, math.nan, dtype=torch.float64)


def _reshaped(s, old, new):
    """Sizes `s` (of a value of shape `old`, dims of 1 where alike) as sizes of
    the same value reshaped to `new`."""
    if not all(old) or not all(new):
        return None
    source, target, i, j = [], [], 0, 0
    while i < len(old) or j < len(new):
        # the next groups of dims with the same number of elements
        i0, j0 = i, j
        a, b = (old[i] if i < len(old) else 1), (new[j] if j < len(new) else 1)
        i, j = min(i + 1, len(old)), min(j + 1, len(new))
        while a != b:
            if a < b:
                a, i = a * old[i], i + 1
            else:
                b, j = b * new[j], j + 1
        alike = all(s.shape[d] == 1 for d in range(i0, i))
        source += [1] * (i - i0) if alike else list(old[i0:i])
        target += [1] * (j - j0) if alike else list(new[j0:j])
    return s.expand(source).reshape(target)
