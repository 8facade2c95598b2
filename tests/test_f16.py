"""fp32 products on fp16 pairs, on the CPU: the pair copies of weights, the
bounds that make a fixed activation scale safe, which products take the path,
and the plan's meaning through the host interpreter."""

import copy

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import kiln
import oracle
from kiln.hip import autotune, f16
from kiln.hip import lib as kl
from kiln.hip.bounds import Bounds
from kiln.hip.lowering import _Lowerer, lower_graph, operand_scales
from models.transformer import Block, gpt2_init_
from test_interpret import check
from test_lowering import lowered


@pytest.fixture
def interpreting(monkeypatch):
    monkeypatch.setenv("KILN_HIP_INTERPRET", "1")


def decode(copy, scales):
    b, n, kp = copy.shape
    copy, scales = copy.numpy(), scales.numpy()
    h = copy.view(np.float16).reshape(b, n, kp // 8, 2, 8).astype(np.float64)
    return (h[:, :, :, 0] + h[:, :, :, 1]).reshape(b, n, kp) * scales.astype(np.float64)[:, :, None]


@pytest.mark.parametrize("k,n", [(8, 3), (40, 24), (61, 5), (768, 2)])
def test_pair_copy_holds_23_bits_per_column(k, n):
    # each column its own power of two: columns 2^-40 .. 2^30 in size keep the
    # relative precision of their largest weights (half an ulp of l: 2^-23 of
    # the value, 2^-25 of 2^-14 of the column's largest below that)
    w = np.random.default_rng(0).standard_normal((k, n)).astype(np.float32)
    w *= (2.0 ** np.linspace(-40, 30, n)).astype(np.float32)
    if n > 3:
        w[:, 3] = 0.0
    args = (w, 0, (0, n, 1), 1, k, n)
    got = decode(f16.pair_rows(*args), f16.column_scales(*args, 0))[0, :, :k].T
    top = np.abs(w).max(axis=0)
    assert (np.abs(got - w) <= 2.0 ** -23 * np.abs(w) + 2.0 ** -39 * top).all()
    assert (f16.pair_rows(*args).reshape(n, -1)[:, f16.padded_k(k):] == 0).all()
    assert torch.equal(f16.column_scales(*args, 5), f16.column_scales(*args, 0) / 32)


def _bounds(model, x):
    g, _ = lowered(model, x, fuse_attention=True)
    return g, _Lowerer(g, "fp32", None)


@pytest.mark.parametrize("scale", [1e-6, 1.0, 1e6])
def test_bounds_hold_whatever_the_input(scale):
    # LayerNorm -> Linear -> GELU -> Linear: every product's A operand stays
    # under its bound, for inputs of any size and rows with one outlier
    torch.manual_seed(1)
    ln, fc, proj = torch.nn.LayerNorm(64), torch.nn.Linear(64, 256), torch.nn.Linear(256, 64)
    torch.nn.init.normal_(ln.weight, 1.0, 0.5), torch.nn.init.normal_(ln.bias)
    model = torch.nn.Sequential(ln, fc, torch.nn.GELU(), proj).eval()
    x = torch.randn(300, 64) * scale
    x[7] = 0.0
    x[7, 3] = 1e5 * scale
    g, low = _bounds(model, x)
    tops = [low.bounds.largest(next(n for n in k.nodes if n.op == "matmul").inputs[0]) for k in g.kernels
            if k.kind == "matmul"]
    with torch.no_grad():
        a = ln(x)
        b = F.gelu(fc(a))
    assert len(tops) == 2 and float(a.abs().max()) <= tops[0] and float(b.abs().max()) <= tops[1]
    assert float(ln(x).abs().max()) > tops[0] / 64   # not vacuous
    for top in tops:
        assert top * 2.0 ** f16.activation_exponent(top) <= 2.0 ** f16.TOP


class SelfAttention(torch.nn.Module):
    """LayerNorm -> q, k, v (one product) -> attention, heads merged."""

    def __init__(self, d, heads):
        super().__init__()
        self.heads, self.ln, self.qkv = heads, torch.nn.LayerNorm(d), torch.nn.Linear(d, 3 * d)

    def forward(self, x):
        t, c = x.shape
        q, k, v = (y.view(t, self.heads, c // self.heads).transpose(0, 1) for y in self.qkv(self.ln(x)).split(c, dim=1))
        y = F.softmax((q @ k.transpose(-2, -1)) * 0.125, dim=-1) @ v
        return y.transpose(0, 1).contiguous().view(t, c)


def test_bounds_refuse_what_has_none():
    assert f16.activation_exponent(float("inf")) is None and f16.activation_exponent(0.0) is None
    assert f16.activation_exponent(1e30) is None
    # a graph input, and a LayerNorm with a non-finite parameter
    g, low = _bounds(torch.nn.Linear(64, 64).eval(), torch.randn(300, 64))
    assert low.bounds.largest(g.args[0]) == float("inf")
    ln = torch.nn.LayerNorm(64)
    with torch.no_grad():
        ln.weight[3] = float("inf")
    g, prog = lowered(torch.nn.Sequential(ln, torch.nn.Linear(64, 64)).eval(), torch.randn(300, 64))
    assert not any("f16x3" in l.summary for l in prog.launches)


def test_which_products_run_on_pairs():
    g, prog = lowered(Block(768, 12, 512), torch.randn(512, 768), fuse_attention=True)
    matmuls = [l for l in prog.launches if "matmul" in l.name]
    assert len(matmuls) == 4 and all(" f16x3" in l.summary for l in matmuls)
    assert "out:f16" in prog.launches[0].summary and "out:f16" in prog.launches[2].summary
    # T = 128: the products with a LayerNorm prologue stay fp32
    g, prog = lowered(Block(768, 12, 128), torch.randn(128, 768), fuse_attention=True)
    for l in prog.launches:
        if "matmul" in l.name:
            assert ("f16x3" in l.summary) != ("prologue: layernorm" in l.summary)
    # a graph input as A, and a LayerNorm output that is also a result
    ln, lin = torch.nn.LayerNorm(64).eval(), torch.nn.Linear(64, 96).eval()
    for fn in (lambda t: lin(t), lambda t: (lin(ln(t)), ln(t))):
        g, prog = lowered(fn, torch.randn(300, 64))
        assert not any("f16x3" in l.summary for l in prog.launches)


def test_plan_key_follows_the_scales():
    # the scales are the only thing a plan takes from constants' values
    lin = torch.nn.Sequential(torch.nn.LayerNorm(64), torch.nn.Linear(64, 96)).eval()
    x = torch.randn(300, 64)
    g1, p1 = lowered(lin, x)
    with torch.no_grad():
        lin[0].weight.mul_(100.0)
    g2, p2 = lowered(lin, x)
    assert operand_scales(g1) != operand_scales(g2)
    assert p1.launches[-1].desc.fparams[0] != p2.launches[-1].desc.fparams[0]


@pytest.mark.parametrize("T", [40, 300])
def test_interpreted_block(interpreting, T):
    model = gpt2_init_(Block(64, 2, T), seed=0).eval()
    x = torch.randn(T, 64)
    c = kiln.compile(model, (x,), device="cuda")
    assert any("f16x3" in l.summary for l in c._exe.program.launches)
    ref = oracle.block(x.numpy(), {k: v.numpy() for k, v in model.state_dict().items()}, 2)
    np.testing.assert_allclose(c(x).numpy(), ref, rtol=1e-4, atol=1e-5)


def test_interpreted_batched_weights(interpreting):
    class Batched(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.ln, self.w = torch.nn.LayerNorm(96), torch.nn.Parameter(torch.randn(3, 96, 50) * 0.1)

        def forward(self, t):
            return self.ln(t) @ self.w

    c = check(Batched().eval(), torch.randn(3, 300, 96))
    assert any("f16x3" in l.summary for l in c._exe.program.launches)


def test_callers_configuration_on_pairs():
    # a caller may name a pair configuration; where the product cannot run on
    # pairs it is a configuration of another precision like any other
    tile = 102
    cfg = lambda *_: {"tile": tile, "splitk": 1}
    ln, lin = torch.nn.LayerNorm(64).eval(), torch.nn.Linear(64, 96).eval()
    from kiln.api import Options, build_passes
    from kiln.passes.manager import PassManager
    from test_gpu import imported

    for fn, on_pairs in ((lambda t: lin(ln(t)), True), (lambda t: lin(t), False)):
        g = imported(fn, (torch.randn(300, 64),))
        PassManager(build_passes(Options())).run(g)
        prog = lower_graph(g, matmul_config=cfg)
        assert (f"tile {tile} splitk 1 f16x3" in prog.launches[-1].summary) == on_pairs
    assert autotune.PRECISION[tile] == "f16x3"


# -- products whose bound lies far above their values -----------------------------------------


def _chain(n, width, activation, kaiming):
    layers = [torch.nn.LayerNorm(width)]
    for _ in range(n):
        lin = torch.nn.Linear(width, width)
        if kaiming:
            torch.nn.init.kaiming_normal_(lin.weight, nonlinearity="relu")
        layers += [lin] + ([activation()] if activation else [])
    return torch.nn.Sequential(*layers, torch.nn.Linear(width, width)).eval()


def _errors(model, x):
    """Relative errors against float64 of the compiled model and of eager
    fp32, and the number of products on pairs."""
    c = kiln.compile(model, (x,), device="cuda")
    with torch.no_grad():
        got, eager, ref = c(x).double(), model(x).double(), copy.deepcopy(model).double()(x.double())
    pairs = sum("f16x3" in l.summary for l in c._exe.program.launches)
    return *(float((t - ref).norm() / ref.norm()) for t in (got, eager)), pairs


@pytest.mark.parametrize("activation,kaiming", [(torch.nn.GELU, False), (torch.nn.ReLU, True), (None, False)])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 8, 10, 12])
def test_deep_chains_are_as_precise_as_eager(interpreting, n, activation, kaiming):
    # the bound grows by sqrt(width) per product, the values do not: products
    # far from the LayerNorm stay off pairs (on pairs: 0.3 to 1.0 at n = 10)
    torch.manual_seed(n)
    err, eager, pairs = _errors(_chain(n, 64, activation, kaiming), torch.randn(40, 64))
    assert err <= eager
    assert 1 <= pairs <= 4


@pytest.mark.parametrize("outlier", [1e2, 1e4, 1e6, 1e12])
@pytest.mark.parametrize("where", ["gain", "unused gain", "weight", "hidden column"])
def test_outliers_keep_the_other_values_precise(interpreting, outlier, where):
    # one gain, weight or hidden column of another size, taken back by what
    # follows it: it sets the scale that all the others share
    torch.manual_seed(0)
    ln, fc, proj = torch.nn.LayerNorm(64), torch.nn.Linear(64, 64), torch.nn.Linear(64, 64)
    with torch.no_grad():
        if where == "gain":
            ln.weight[0] = outlier
            fc.weight[:, 0] /= outlier
        elif where == "unused gain":
            ln.weight[0] = outlier
            fc.weight[:, 0] = 0.0
        elif where == "weight":
            ln.weight[0] = 0.1 / outlier
            fc.weight[:, 0] *= outlier
        else:
            fc.weight[0] *= outlier
            proj.weight[:, 0] /= outlier
    err, eager, _ = _errors(torch.nn.Sequential(ln, fc, proj).eval(), torch.randn(300, 64))
    assert err <= eager


def test_columns_out_of_the_scales_range_stay_off_pairs(interpreting):
    # a column's power of two is clamped: weights below 2^-66 would be fp16
    # subnormals. And bounds whose squares vanish in fp32 are still bounds.
    torch.manual_seed(0)
    ln, fc, proj = torch.nn.LayerNorm(64), torch.nn.Linear(64, 64, bias=False), torch.nn.Linear(64, 64)
    with torch.no_grad():
        fc.weight *= 1e-25
    err, eager, pairs = _errors(torch.nn.Sequential(ln, fc).eval(), torch.randn(300, 64))
    assert err <= eager and pairs == 0
    with torch.no_grad():
        ln.weight *= 1e24
    g, low = _bounds(torch.nn.Sequential(ln, fc, proj).eval(), torch.randn(300, 64))
    mm = [n for n in g.nodes if n.op == "matmul"][-1]
    with torch.no_grad():
        hidden = fc(ln(torch.randn(300, 64)))
    assert float(hidden.abs().max()) <= low.bounds.largest(mm.inputs[0]) < float("inf")


@pytest.mark.parametrize("scale_q,scale_v,on_pairs", [(1.0, 1.0, True), (64.0, 8.0, True), (1e5, 1.0, False),
                                                      (1.0, 1e-5, False)])
def test_attention_on_pairs_needs_tight_bounds(scale_q, scale_v, on_pairs):
    # a head of another size shares the others' scale
    torch.manual_seed(0)
    model = SelfAttention(128, 2).eval()
    with torch.no_grad():
        model.qkv.weight[:64] *= scale_q
        model.qkv.weight[256 + 64:] *= scale_v
        model.qkv.bias[:64] *= scale_q
        model.qkv.bias[256 + 64:] *= scale_v
    g, prog = lowered(model, torch.randn(200, 128), fuse_attention=True)
    assert any("products:f16x3" in l.summary for l in prog.launches) == on_pairs


@pytest.mark.parametrize("T,d,heads", [(512, 768, 12), (2048, 768, 12), (2048, 1024, 16), (333, 128, 4)])
def test_blocks_are_tight(T, d, heads):
    # the bounds of a block lie close enough for all its products and attention
    g, prog = lowered(gpt2_init_(Block(d, heads, T), seed=0), torch.randn(T, d), fuse_attention=True)
    assert sum("f16x3" in l.summary for l in prog.launches) == 5


def test_sizes_follow_the_graph():
    # measured rows against the sizes the gate works with: a LayerNorm's per
    # column, through a product, GELU, views and attention to a small factor
    torch.manual_seed(0)
    model = SelfAttention(128, 2).eval()
    with torch.no_grad():
        model.ln.weight.uniform_(0.2, 3.0), model.ln.bias.uniform_(-0.5, 0.5)
    x = torch.randn(200, 128)
    g, low = _bounds(model, x)
    (kernel,) = [k for k in g.kernels if k.kind == "attention"]
    m = low._attention_match(kernel)
    with torch.no_grad():
        q, k, v = (t.view(200, 2, 64).transpose(0, 1) for t in model.qkv(model.ln(x)).split(128, dim=1))
    for value, data in ((m.q, q), (m.v, v)):
        ratio = data.double().square().mean(dim=-2, keepdim=True).sqrt() / low.bounds.size(value)
        assert ratio.shape == (2, 1, 64) and 0.7 < float(ratio.min()) and float(ratio.max()) < 1.4
    assert torch.isnan(low.bounds.size(g.args[0])).all()


# -- storage of operands that are read another way too ------------------------------------------


class _ResidualOnNorm(torch.nn.Module):
    """y + W y of y = LayerNorm(x): the product's A operand is its residual."""

    def __init__(self, d, view):
        super().__init__()
        self.ln, self.lin, self.view = torch.nn.LayerNorm(d), torch.nn.Linear(d, d), view

    def forward(self, x):
        y = self.ln(x)
        if self.view:   # the residual through a view of the same buffer
            return self.lin(y) + y.view(2, x.shape[0] // 2, -1).transpose(0, 1).transpose(0, 1).reshape(x.shape)
        return self.lin(y) + y


@pytest.mark.parametrize("precision", ["fp32", "bf16", "bf16x3"])
@pytest.mark.parametrize("T,d,tile", [(300, 64, None), (600, 64, None), (600, 256, 98), (40, 64, None)])
@pytest.mark.parametrize("view", [False, True])
def test_operand_that_is_also_the_residual_stays_fp32(interpreting, precision, T, d, tile, view):
    torch.manual_seed(0)
    cfg = {"gpu_matmul_config": lambda *_: {"tile": tile, "splitk": 1}} if tile is not None and precision == "bf16" else {}
    c = check(_ResidualOnNorm(d, view).eval(), torch.randn(T, d), matmul_precision=precision, **cfg,
              **({} if precision == "fp32" else {"rtol": 2e-2, "atol": 2e-2}))
    product = c._exe.program.launches[-1].desc
    assert product.cfg[7] & 1 == 0 and product.cfg[7] >> 16 & 1 == 0


# -- stored plans -------------------------------------------------------------------------------


class _Projected(SelfAttention):
    """SelfAttention with separate q, k and v products and an output projection."""

    def __init__(self, d, heads):
        super().__init__(d, heads)
        self.q, self.k, self.v, self.proj = (torch.nn.Linear(d, d) for _ in range(4))

    def forward(self, x):
        t, c = x.shape
        y = self.ln(x)
        q, k, v = (f(y).view(t, self.heads, c // self.heads).transpose(0, 1) for f in (self.q, self.k, self.v))
        y = F.softmax((q @ k.transpose(-2, -1)) * 0.125, dim=-1) @ v
        return self.proj(y.transpose(0, 1).contiguous().view(t, c))


def _descs(program):
    return [bytes(l.desc) for l in program.launches]


@pytest.mark.parametrize("change", [
    ("qkv", 4096.0), ("qkv", 2.0 ** -12), ("one head", 1e6), ("q", 4096.0), ("v", 4096.0), ("v", 2.0 ** -12),
    ("column", 1e-25)])
def test_stored_plan_is_not_reused_with_other_scales(interpreting, tmp_path, monkeypatch, change):
    # two models of one structure against one cache: the second's plan has
    # the scales, and the storage, that a fresh lowering gives it
    monkeypatch.setenv("KILN_CACHE_DIR", str(tmp_path))
    what, factor = change
    torch.manual_seed(0)
    model = (_Projected if what in ("q", "v", "column") else SelfAttention)(64, 2 if what != "qkv" else 1).eval()
    x = torch.randn(192, 64)
    first = kiln.compile(model, (x,), device="cuda")
    assert any("products:f16x3" in l.summary for l in first._exe.program.launches)
    again = kiln.compile(model, (x,), device="cuda")
    assert again.report.lowering["plan_cache"] == "stored"
    with torch.no_grad():
        if what == "one head":
            model.qkv.weight[:32] *= factor
        elif what == "column":
            model.proj.weight[0] *= factor
        else:
            getattr(model, what).weight.mul_(factor)
    second = kiln.compile(model, (x,), device="cuda")
    fresh = kiln.compile(model, (x,), device="cuda", plan_cache=False)
    assert _descs(second._exe.program) == _descs(fresh._exe.program) != _descs(first._exe.program)
    assert second.report.lowering["plan_cache"] == "lowered"


class _Masked(SelfAttention):
    def __init__(self, d, heads, mask):
        super().__init__(d, heads)
        self.register_buffer("mask", mask)

    def forward(self, x):
        t, c = x.shape
        q, k, v = (y.view(t, self.heads, c // self.heads).transpose(0, 1) for y in self.qkv(self.ln(x)).split(c, dim=1))
        y = F.softmax(q @ k.transpose(-2, -1) * 0.2 + self.mask, dim=-1) @ v
        return y.transpose(0, 1).contiguous().view(t, c)


@pytest.mark.parametrize("precision", ["fp32", "bf16x3", "bf16"])
@pytest.mark.parametrize("T", [1, 40])
def test_stored_plan_is_not_reused_with_another_mask(interpreting, tmp_path, monkeypatch, precision, T):
    # a causal mask is not read by its plan; another mask of the same shape is
    monkeypatch.setenv("KILN_CACHE_DIR", str(tmp_path))
    causal = torch.full((T, T), float("-inf")).triu(1)
    x = torch.randn(T, 64)
    for mask in (causal, torch.randn(T, T) if T > 1 else torch.full((1, 1), float("-inf")), causal):
        torch.manual_seed(0)
        model = _Masked(64, 2, mask).eval()
        c = kiln.compile(model, (x,), device="cuda", matmul_precision=precision)
        with torch.no_grad():
            torch.testing.assert_close(c(x), model(x), rtol=3e-2, atol=3e-2, equal_nan=True)
    assert c.report.lowering["plan_cache"] == "stored"


@pytest.mark.parametrize("batch,k,n", [(1, 40, 24), (3, 61, 5), (2, 8, 1)])
@pytest.mark.parametrize("chunk", [1, 64, 200])
def test_pair_copy_in_chunks_has_the_same_bits(batch, k, n, chunk):
    # a transposed view at an offset, made whole and a few rows at a time;
    # exponents and scales come from the same read of the weight
    w = np.random.default_rng(1).standard_normal(7 + batch * k * n).astype(np.float32)
    args = (w, 7, (k * n, 1, k), batch, k, n)
    copy, exponents = f16.pair_copy(*args, chunk=chunk)
    assert torch.equal(copy, f16.pair_rows(*args))
    assert torch.equal(exponents, f16.column_exponents(*args))
    assert torch.equal(f16.scales_of(exponents, 3), f16.column_scales(*args, 3))


# -- what the pair configurations refuse --------------------------------------------------------


@pytest.mark.parametrize("m,on_pairs", [(699050, True), (699051, False)])
def test_operands_of_2_29_elements_stay_off_pairs(m, on_pairs):
    # rows of 768: (m - 1) * 768 + 768 below 2^29, the library's limit for
    # 32-bit byte offsets, and above
    from kiln.api import Options, build_passes
    from kiln.passes.manager import PassManager

    w, b = np.full((768, 64), 0.02, np.float32), np.zeros(64, np.float32)
    g = autotune._linear_graph(1, m, 64, 768, w, b, True)
    PassManager(build_passes(Options())).run(g)
    prog = lower_graph(g)
    assert ("f16x3" in prog.launches[-1].summary) == on_pairs
    if not on_pairs:
        kl.Plan([l.desc for l in prog.launches])   # the library takes it


@pytest.mark.parametrize("residuals,on_pairs", [(7, True), (8, False)])
def test_epilogue_that_fills_the_operand_table_stays_off_pairs(interpreting, residuals, on_pairs):
    # a launch has 12 operands: the product's two, bias, residuals, output,
    # and on pairs the column scales
    torch.manual_seed(0)
    ln, lin = torch.nn.LayerNorm(64).eval(), torch.nn.Linear(64, 48).eval()

    def fn(x, *rs):
        y = lin(ln(x))
        for r in rs:
            y = y + r
        return y

    c = check(fn, torch.randn(300, 64), *[torch.randn(300, 48) for _ in range(residuals)])
    assert any("f16x3" in l.summary for l in c._exe.program.launches) == on_pairs


# -- what the host interpreter sees of pairs ------------------------------------------------------


@pytest.mark.parametrize("q,v", [(1.0, 1.0), (32.0, 32.0), (2.0 ** -9, 2.0 ** -12), (2.0 ** 9, 2.0 ** 12)])
def test_interpreted_attention_on_pairs(interpreting, q, v):
    # q and k of very different size (the scores stay), v large and small: each
    # in its own buffer with its own scale
    torch.manual_seed(0)
    model = _Projected(64, 2).eval()
    with torch.no_grad():
        for lin, s in ((model.q, q), (model.k, 1.0 / q), (model.v, v)):
            lin.weight.mul_(s), lin.bias.mul_(s)
    c = kiln.compile(model, (torch.randn(192, 64),), device="cuda")
    assert any("products:f16x3" in l.summary for l in c._exe.program.launches)
    err, eager, _ = _errors(model, torch.randn(192, 64))
    assert err <= eager


@pytest.mark.parametrize("factor,loses", [(4096.0, "range"), (2.0 ** -45, "bits")])
def test_interpreter_sees_stale_scales(interpreting, tmp_path, monkeypatch, factor, loses):
    # a plan with another model's scales of q, k and v: values past fp16's
    # range are not finite, values far below it lose their bits
    from kiln.hip import lowering

    monkeypatch.setenv("KILN_CACHE_DIR", str(tmp_path))
    monkeypatch.setattr(lowering, "constant_facts", lambda *_: "")
    torch.manual_seed(0)
    model, x = SelfAttention(64, 2).eval(), torch.randn(192, 64)
    kiln.compile(model, (x,), device="cuda")
    with torch.no_grad():
        model.qkv.weight[128:] *= factor
        model.qkv.bias[128:] *= factor
    c = kiln.compile(model, (x,), device="cuda")
    assert c.report.lowering["plan_cache"] == "stored"
    out = c(x)
    with torch.no_grad():
        ref = copy.deepcopy(model).double()(x.double())
    if loses == "range":
        assert not torch.isfinite(out).all()
    else:
        assert float((out.double() - ref).norm() / ref.norm()) > 1e-3
    monkeypatch.undo()
    monkeypatch.setenv("KILN_HIP_INTERPRET", "1")
    fresh = kiln.compile(model, (x,), device="cuda", plan_cache=False)(x)
    assert float((fresh.double() - ref).norm() / ref.norm()) < 1e-6


# -- rows far smaller than usual ------------------------------------------------------------------


@pytest.mark.parametrize("spread", [1.0, 1e-3, 1e-5, 1e-6, 1e-7, 1e-8, 1e-9])
@pytest.mark.parametrize("what", ["linear", "mlp", "values"])
def test_small_rows_keep_their_precision(interpreting, spread, what):
    # a LayerNorm's rows shrink where their spread is small against sqrt(eps)
    # = 3e-3, and without biases so does everything behind them; the scale is
    # one for all rows. (1e-9: 2^-21 of the usual size.)
    torch.manual_seed(0)
    if what == "values":
        model = SelfAttention(64, 2)
        torch.nn.init.zeros_(model.qkv.bias)
    else:
        layers = [torch.nn.LayerNorm(64), torch.nn.Linear(64, 64, bias=False)]
        model = torch.nn.Sequential(*layers, *([torch.nn.GELU(), torch.nn.Linear(64, 64, bias=False)] if what == "mlp" else []))
    err, eager, pairs = _errors(model.eval(), torch.randn(300, 64) * spread)
    assert err <= eager and pairs >= 1


@pytest.mark.parametrize("rows,k,on_pairs", [(1025, 96, False), (1025, 128, True), (1024, 96, True)])
def test_shallow_products_of_many_rows_stay_off_pairs(rows, k, on_pairs):
    # (lower error on the fp32 tiles there)
    model = torch.nn.Sequential(torch.nn.LayerNorm(k), torch.nn.Linear(k, 64)).eval()
    _, prog = lowered(model, torch.randn(rows, k))
    assert ("f16x3" in prog.launches[-1].summary) == on_pairs
