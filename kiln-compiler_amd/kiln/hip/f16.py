"""fp16-pair copies of GEMM weights (fp32 products on the fp16 matrix cores).

A weight x is held as h = fp16(x * 2^e) and l = fp16(x * 2^e - h): 23 of its
24 significant bits, and 2^-39 of its column's largest weight below
(csrc/kh_common.hpp; kiln/hip/bounds.py says which products take them). The library reads B as [batch][N][K']
rows (K' = K rounded up to 8, zero padded), in blocks of 8 values: 16 bytes of
h, then 16 bytes of l. Each output column n has its own power of two, which
puts the column's largest weight just below 2^15; the product's epilogue
multiplies by ``column_scales``, one exact power of two per column that takes
back the weights' scale and the activations'.
"""

from __future__ import annotations

import math

import numpy as np
import torch

# the largest scaled magnitude is below 2^TOP: fp16's largest finite value is
# 65504, and a bound on activations may be missed by rounding
TOP = 14
# exponents that keep every scale and product of scales a normal float32
WEIGHT_EXPONENTS = (-80, 80)
ACTIVATION_EXPONENTS = (-40, 40)
# elements of a pair copy that are made at a time (temporaries of ~100 MB)
CHUNK = 4 << 20


def activation_exponent(bound: float):
    """e with bound * 2^e <= 2^TOP for activations of magnitude <= bound, or
    None when the bound is no use (not finite, or its scale out of range)."""
    if not math.isfinite(bound) or bound <= 0.0:
        return None
    e = TOP - math.ceil(math.log2(bound))
    low, high = ACTIVATION_EXPONENTS
    return e if low <= e <= high else None


def padded_k(k: int) -> int:
    return (k + 7) // 8 * 8


def _rows(data: np.ndarray, offset: int, strides, batch: int, k: int, n: int, device) -> torch.Tensor:
    """The [batch, K, N] view (element offset, strides over (b, k, n)) of a
    constant as float32 [batch, N, K] on `device` (a view)."""
    flat = torch.from_numpy(np.ascontiguousarray(data, dtype=np.float32).reshape(-1)).to(device)
    sb, sk, sn = (int(s) for s in strides)
    return torch.as_strided(flat, (batch, n, k), (sb, sn, sk), offset)


def row_exponents(rows: torch.Tensor) -> torch.Tensor:
    """e [batch, N] (int32) of float32 [batch, N, K]: a row's largest magnitude
    times 2^e lands in [2^TOP, 2^(TOP + 1))."""
    top = torch.maximum(rows.amax(dim=-1), -rows.amin(dim=-1))
    _, exponent = torch.frexp(top)   # top in [2^(exponent - 1), 2^exponent)
    return torch.where(top > 0, TOP + 1 - exponent, torch.zeros_like(exponent)).clamp(*WEIGHT_EXPONENTS)


def columns_fit(top: torch.Tensor) -> bool:
    """Is no column's power of two (largest weights ``top``) out of range?"""
    _, exponent = torch.frexp(top[top > 0])
    e = TOP + 1 - exponent
    return not e.numel() or (int(e.min()) >= WEIGHT_EXPONENTS[0] and int(e.max()) <= WEIGHT_EXPONENTS[1])


def _power_of_two(e: torch.Tensor) -> torch.Tensor:
    """float32 2^e, |e| <= 126, from its bits (torch.ldexp goes through pow,
    which the GPU does not round to an exact power)."""
    return ((e.int() + 127) << 23).view(torch.float32)


def column_exponents(data, offset, strides, batch: int, k: int, n: int, device="cpu") -> torch.Tensor:
    """The exponents of the powers of two of the [batch, K, N] view's columns
    (int32 [batch, N], on `device`)."""
    return row_exponents(_rows(data, offset, strides, batch, k, n, device))


def pair_rows(data, offset, strides, batch: int, k: int, n: int, device="cpu", chunk=CHUNK) -> torch.Tensor:
    """The pair copy alone (see pair_copy)."""
    return pair_copy(data, offset, strides, batch, k, n, device, chunk)[0]


def pair_copy(data, offset, strides, batch: int, k: int, n: int, device="cpu", chunk=CHUNK):
    """(the [batch, N, K'] pair copy (int32 words, on `device`) of the [batch, K,
    N] view of a constant, each row times its own power of two; the exponents
    of those, as column_exponents gives them). The same bits on the CPU and on
    the GPU, where it is ~100 times faster. Made a few rows at a time, `chunk`
    elements: beside the result and the constant itself it takes
    scratch_bytes."""
    source = _rows(data, offset, strides, batch, k, n, device)
    kp = padded_k(k)
    out = torch.empty((batch, n, kp // 8, 2, 8), dtype=torch.float16, device=device)
    exponents = torch.empty((batch, n), dtype=torch.int32, device=device)
    step = max(1, chunk // kp)
    for b in range(batch):
        for at in range(0, n, step):
            rows = source[b, at:at + step].contiguous()
            e = exponents[b, at:at + step] = row_exponents(rows)
            rows = rows * _power_of_two(e).unsqueeze(-1)
            if kp != k:
                rows = torch.nn.functional.pad(rows, (0, kp - k))
            rows = rows.view(-1, kp // 8, 8)
            h = rows.half()   # (rounds to nearest)
            out[b, at:at + step, :, 0] = h
            out[b, at:at + step, :, 1] = (rows - h.float()).half()
    return out.view(torch.int32).view(batch, n, kp), exponents


def column_scales(data, offset, strides, batch: int, k: int, n: int, activation_e: int, device="cpu") -> torch.Tensor:
    """2^-(e + activation_e) per column (float32 [batch, N]): what a product of
    the scaled operands is multiplied by."""
    return scales_of(column_exponents(data, offset, strides, batch, k, n, device), activation_e)


def scales_of(exponents: torch.Tensor, activation_e: int) -> torch.Tensor:
    return _power_of_two(-(exponents + activation_e))


def scratch_bytes(elements: int, batch: int, k: int, n: int) -> int:
    """Device memory that making a pair copy of a view of a constant of so many
    elements takes beside the copy: the constant, at most six fp32 values per
    element of a chunk, and per row a few words."""
    kp = padded_k(k)
    return 4 * elements + 24 * min(max(CHUNK, kp), batch * n * kp) + 64 * batch * n


def pair_bytes(batch: int, k: int, n: int) -> int:
    return 4 * batch * n * padded_k(k)
