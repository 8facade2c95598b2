"""Parity of the fp32 products on fp16 pairs (tiles of precision "f16x3"):
against float64 of the fp32 inputs at the fp32 suite's tolerance, and with an
error no larger than an fp32 MFMA configuration's that sums K in one chain."""

import copy

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import kiln
import oracle
from kiln.hip import autotune
from models.transformer import Block, gpt2_init_
from test_gpu import ATOL, RTOL

pytestmark = pytest.mark.gpu

TILES = [t for t in sorted(autotune.TILES) if autotune.PRECISION[t] == "f16x3"]
FP32_CHAIN = 4   # the fp32 copy pipeline's 32x64 tile


class _LnLinear(torch.nn.Module):
    """LayerNorm -> Linear, then an epilogue: none, "res" (residual), an
    activation, or "tape" (one that the direct epilogue does not have)."""

    def __init__(self, k, n, epilogue):
        super().__init__()
        self.ln, self.lin, self.epilogue = torch.nn.LayerNorm(k), torch.nn.Linear(k, n), epilogue
        with torch.no_grad():
            self.lin.weight.normal_(0.0, 1.0 / k ** 0.5)
            self.ln.weight.normal_(1.0, 0.3), self.ln.bias.normal_(0.0, 0.3)

    def forward(self, x, r):
        y = self.lin(self.ln(x))
        if self.epilogue == "res":
            return y + r
        if self.epilogue == "tape":
            return torch.tanh(y) * r
        return F.gelu(y, approximate=self.epilogue) if self.epilogue in ("tanh", "none") else y


def _run(model, args, tile):
    c = kiln.compile(model, args, device="cuda", cuda_graphs=False,
                     gpu_matmul_config=lambda *_: {"tile": tile, "splitk": 1})
    return c, c(*args)


# M and N around and between tile edges, K from one step to more than the ring
# holds, odd and even step counts
SHAPES = [(1100, 200, 32, "res"), (1030, 133, 64, "linear"), (1027, 8, 96, "tanh"), (1153, 452, 160, "none"),
          (1061, 97, 768, "tape"), (1025, 384, 224, "res")]


@pytest.mark.parametrize("tile", TILES)
def test_every_pair_configuration(tile):
    for m, n, k, epilogue in SHAPES:
        if tile in autotune.SMALL_M:
            m -= 1020     # 5 .. 133 rows
        torch.manual_seed(m + n + k)
        model = _LnLinear(k, n, epilogue).eval()
        args = (torch.randn(m, k) * 3 + 1, torch.randn(m, n))
        print(tile, m, n, k, epilogue, flush=True)
        c, out = _run(model, args, tile)
        assert f"tile {tile} splitk 1 f16x3" in c._exe.program.launches[-1].summary
        _, plain = _run(model, args, FP32_CHAIN)
        with torch.no_grad():
            ref = model.double()(*(t.double() for t in args))
        np.testing.assert_allclose(out.cpu().double().numpy(), ref.numpy(), rtol=RTOL, atol=ATOL)
        err, err_plain = ((t.cpu().double() - ref).norm() / ref.norm() for t in (out, plain))
        # (a few roundings at K = 32: the two agree to a factor)
        assert err <= (1.1 if k > 96 else 1.5) * err_plain + 1e-9, (err, err_plain)
        for _ in range(3):
            assert torch.equal(c(*args), out)


def test_pair_copies_made_on_the_gpu_have_the_cpus_bits():
    from kiln.hip import f16

    w = np.random.default_rng(0).standard_normal((77, 133)).astype(np.float32) * np.logspace(-9, 5, 133, dtype=np.float32)
    args = (w, 0, (0, 133, 1), 1, 77, 133)
    assert torch.equal(f16.pair_rows(*args, "cuda").cpu(), f16.pair_rows(*args))
    assert torch.equal(f16.column_scales(*args, 3, "cuda").cpu(), f16.column_scales(*args, 3))


def test_columns_of_very_different_size_keep_their_precision():
    torch.manual_seed(3)
    model = _LnLinear(256, 96, "linear").eval()
    with torch.no_grad():
        model.lin.weight *= (10.0 ** torch.linspace(-8, 4, 96))[:, None]
        model.lin.bias.zero_()
    args = (torch.randn(300, 256), torch.randn(300, 96))
    _, out = _run(model, args, 102)
    with torch.no_grad():
        ref = model.double()(*(t.double() for t in args))
    err = (out.cpu().double() - ref).norm(dim=0) / ref.norm(dim=0)
    assert float(err.max()) <= 5e-7     # 24 steps' roundings; a shared scale would lose the small columns


@pytest.mark.parametrize("loc,scale", [(0.0, 1e-4), (100.0, 1.0), (0.0, 1e8)])
def test_rows_of_any_size_and_non_finite_rows(loc, scale):
    torch.manual_seed(4)
    model = _LnLinear(128, 200, "linear").eval()
    x = torch.randn(300, 128) * scale + loc
    bad = [3, 64, 299]
    for row, v in zip(bad, (float("nan"), float("inf"), -float("inf"))):
        x[row, 5] = v
    args = (x, torch.randn(300, 200))
    _, out = _run(model, args, 103)
    _, plain = _run(model, args, FP32_CHAIN)
    good = [i for i in range(300) if i not in bad]
    assert torch.isnan(out[bad]).all()
    # against the fp32 product on the same LayerNorm rows
    np.testing.assert_allclose(out[good].cpu().numpy(), plain[good].cpu().numpy(), rtol=RTOL, atol=ATOL)


class _Attention(torch.nn.Module):
    """LayerNorm -> q, k, v (one product) -> attention, heads merged."""

    def __init__(self, d, heads, tokens, mask, scale):
        super().__init__()
        self.heads, self.scale = heads, scale
        self.ln, self.qkv = torch.nn.LayerNorm(d), torch.nn.Linear(d, 3 * d)
        with torch.no_grad():
            self.qkv.weight.normal_(0.0, 1.0 / d ** 0.5), self.qkv.bias.normal_(0.0, 0.1)
        if mask == "causal":
            self.register_buffer("mask", torch.full((tokens, tokens), float("-inf")).triu(1))
        elif mask == "add":
            m = torch.randn(tokens, tokens).masked_fill(torch.rand(tokens, tokens) < 0.3, float("-inf"))
            m[5] = float("-inf")     # a row that sees no key: NaN, as in eager
            self.register_buffer("mask", m)
        else:
            self.mask = None

    def forward(self, x):
        t, c = x.shape
        q, k, v = (y.view(t, self.heads, c // self.heads).transpose(0, 1) for y in self.qkv(self.ln(x)).split(c, dim=1))
        s = (q @ k.transpose(-2, -1)) * self.scale
        s = s if self.mask is None else s + self.mask
        return (F.softmax(s, dim=-1) @ v).transpose(0, 1).contiguous().view(t, c)


# keys from the fewest that take the path: whole blocks, one past, one short;
# both head dims; a negative and a zero scale; fully masked rows
@pytest.mark.parametrize("tokens,d,heads,mask,scale", [
    (160, 128, 2, None, 0.125), (161, 128, 4, "causal", 0.17), (191, 64, 2, "causal", 0.17), (192, 64, 1, "add", 0.125),
    (333, 256, 4, "causal", 0.125), (333, 256, 8, "add", 0.17), (257, 128, 2, None, -0.2), (200, 128, 2, "causal", 0.0),
    (1025, 128, 2, "causal", 0.125)])
def test_attention_on_pairs(tokens, d, heads, mask, scale, monkeypatch):
    from kiln.hip import lowering

    torch.manual_seed(tokens)
    model, x = _Attention(d, heads, tokens, mask, scale).eval(), torch.randn(tokens, d)

    def run():
        c = kiln.compile(model, (x,), device="cuda", cuda_graphs=False, plan_cache=False)
        return c, c(x.cuda())

    c, out = run()
    assert any("products:f16x3" in l.summary for l in c._exe.program.launches)
    monkeypatch.setattr(lowering._Lowerer, "f16_attention", lambda self, k: None)
    _, plain = run()
    with torch.no_grad():
        ref = model.double()(x.double())
    out, plain = out.cpu().double(), plain.cpu().double()
    bad = torch.isnan(ref)
    assert torch.equal(torch.isnan(out), bad)
    np.testing.assert_allclose(out[~bad].numpy(), ref[~bad].numpy(), rtol=RTOL, atol=ATOL)
    err, err_plain = ((t - ref)[~bad].norm() / ref[~bad].norm() for t in (out, plain))
    assert err <= 1.1 * err_plain, (err, err_plain)
    for _ in range(3):
        assert torch.equal(c(x.cuda()).cpu().double()[~bad], out[~bad])


@pytest.mark.parametrize("T", [16, 300, 777])
def test_block_on_pairs(T):
    model = gpt2_init_(Block(256, 4, T), seed=0).eval()
    x = torch.randn(T, 256)
    c = kiln.compile(model, (x,), device="cuda")
    assert any("f16x3" in l.summary for l in c._exe.program.launches)
    ref = oracle.block(x.numpy(), {k: v.numpy() for k, v in model.state_dict().items()}, 4)
    np.testing.assert_allclose(c(x.cuda()).cpu().numpy(), ref, rtol=RTOL, atol=ATOL)
    exe = c._exe
    for _ in range(3):     # graph replays, with eager work between them
        exe.replay_only()
        torch.zeros(8, device="cuda").add_(1)
    exe._static[0][0].copy_(x.cuda())
    exe.replay_only()
    assert torch.equal(exe._static[1][0], c(x.cuda()))


@pytest.mark.parametrize("precision,tol", [("fp32", 1e-4), ("bf16x3", 1e-4), ("bf16", 2e-2)])
def test_operand_that_is_also_the_residual(precision, tol):
    from test_f16 import _ResidualOnNorm

    torch.manual_seed(0)
    model, x = _ResidualOnNorm(256, False).eval(), torch.randn(600, 256)
    out = kiln.compile(model, (x,), device="cuda", matmul_precision=precision)(x.cuda()).cpu()
    with torch.no_grad():
        ref = model.double()(x.double())
    np.testing.assert_allclose(out.double().numpy(), ref.numpy(), rtol=tol, atol=tol)


def test_compile_returns_with_its_weights_made():
    # weights are made by kernels of the stream that compiles; calls come on
    # any stream, so nothing may be pending, and what is made beside the copy
    # stays under the size that the memory check counts
    from kiln.hip import f16

    model = torch.nn.Sequential(torch.nn.LayerNorm(1024), torch.nn.Linear(1024, 8192, bias=False)).eval()
    x = torch.randn(300, 1024)
    side = torch.cuda.Stream()
    for stream in (torch.cuda.current_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            c = kiln.compile(model, (x,), device="cuda", cuda_graphs=False)
            assert stream.query()
        xd = x.cuda()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            out = c(xd)
        side.synchronize()
        torch.testing.assert_close(out.cpu(), model(x).detach(), rtol=RTOL, atol=1e-4)
    w = np.ones((1024, 8192), np.float32)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    copy, exponents = f16.pair_copy(w, 0, (0, 8192, 1), 1, 1024, 8192, "cuda")
    peak = torch.cuda.max_memory_allocated() - before
    assert peak <= f16.pair_bytes(1, 1024, 8192) + f16.scratch_bytes(w.size, 1, 1024, 8192)


@pytest.mark.parametrize("spread", [1e-6, 1e-8])
@pytest.mark.parametrize("tile", [101, 102, 103, 106, 107])
def test_small_rows_keep_their_precision(tile, spread):
    # LayerNorm rows 2^-11.6 and 2^-18.3 of the usual size (spread / sqrt(eps))
    torch.manual_seed(5)
    rows = 1100 if tile not in autotune.SMALL_M else 70
    model = torch.nn.Sequential(torch.nn.LayerNorm(256), torch.nn.Linear(256, 200, bias=False)).eval()
    x = torch.randn(rows, 256) * spread
    errs = []
    for t in (tile, FP32_CHAIN):
        c = kiln.compile(model, (x,), device="cuda", cuda_graphs=False,
                         gpu_matmul_config=lambda *_: {"tile": t, "splitk": 1})
        assert ("f16x3" in c._exe.program.launches[-1].summary) == (t == tile)
        ref = copy.deepcopy(model).double()(x.double()).detach()
        errs.append(float((c(x).cpu().double() - ref).norm() / ref.norm()))
    assert errs[0] <= 1.1 * errs[1], errs


@pytest.mark.parametrize("mask", [None, "causal", "add"])
def test_attention_on_small_rows_keeps_its_precision(mask, monkeypatch):
    from kiln.hip import lowering

    torch.manual_seed(6)
    model, x = _Attention(128, 2, 333, mask, 0.125).eval(), torch.randn(333, 128) * 1e-8
    torch.nn.init.zeros_(model.qkv.bias)
    ref = copy.deepcopy(model).double()(x.double()).detach()
    good = ~torch.isnan(ref)

    def err():
        c = kiln.compile(model, (x,), device="cuda", cuda_graphs=False, plan_cache=False)
        out = c(x.cuda()).cpu().double()
        return any("products:f16x3" in l.summary for l in c._exe.program.launches), float(
            (out - ref)[good].norm() / ref[good].norm())

    pairs, on_pairs = err()
    monkeypatch.setattr(lowering._Lowerer, "f16_attention", lambda self, k: None)
    _, plain = err()
    assert pairs and on_pairs <= 1.1 * plain, (on_pairs, plain)


@pytest.mark.parametrize("tokens,heads,mask", [(192, 2, None), (333, 2, "causal"), (200, 4, "causal"), (200, 2, "add")])
@pytest.mark.parametrize("gain", [2.0 ** 9, 2.0 ** 12, 2.0 ** 17])
def test_attention_with_huge_scores(tokens, heads, mask, gain, monkeypatch):
    # scores around gain^2 (up to 2^34, where fp32 tells scores 2^11 apart
    # from equal ones): the softmax is one-hot and finite, as it is in fp32
    from kiln.hip import lowering

    torch.manual_seed(7)
    model, x = _Attention(128, heads, tokens, mask, 0.125).eval(), torch.randn(tokens, 128)
    with torch.no_grad():
        for p in (model.qkv.weight, model.qkv.bias):
            p[:256] *= gain
            p[256:] *= gain      # (v shares the scale: kept as large)
    c = kiln.compile(model, (x,), device="cuda", cuda_graphs=False, plan_cache=False)
    assert any("products:f16x3" in l.summary for l in c._exe.program.launches)
    out = c(x.cuda()).cpu().double()
    monkeypatch.setattr(lowering._Lowerer, "f16_attention", lambda self, k: None)
    plain = kiln.compile(model, (x,), device="cuda", cuda_graphs=False, plan_cache=False)(x.cuda()).cpu().double()
    ref = copy.deepcopy(model).double()(x.double()).detach()
    good = ~torch.isnan(ref)
    assert torch.equal(torch.isfinite(out), good)
    # rows whose two best keys lie apart by more than fp32's rounding of such
    # scores agree; the share of the others is small (2^-10 of a unit's odds)
    row_ok = lambda t: ((t - ref).abs() <= 1e-3 * gain).all(dim=-1) | ~good.all(dim=-1)
    assert float(row_ok(out).float().mean()) >= min(0.97, float(row_ok(plain).float().mean()) - 0.02)
