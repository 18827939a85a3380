"""Infinities, the largest finite values and NaN go where they belong: an
output is infinite or NaN where the same call in float64 (converted to the
call's dtype) is, and only there.

The float32 path multiplies three-plane bf16 splits of its operands, in which
an infinite or nearly infinite operand needs a form of its own. The attention
pass sums the softmax of several queries in one accumulator and recomputes
what leaves the safe range: a query's NaN must stay its own."""

from __future__ import annotations

import dataclasses
import math

import pytest
import torch

from foldjax_amd import kernels
from foldjax_amd import params as P
from foldjax_amd import synthetic as syn
from tests.gpu_util import say

pytestmark = pytest.mark.gpu

INF = math.inf
FLT_MAX = torch.finfo(torch.float32).max
ROUNDS_UP = float.fromhex("0x1.FF8p127")  # finite in float32, past the largest bf16


def _set(w, field, at, value):
    t = getattr(w, field).clone()
    t[at] = value
    return dataclasses.replace(w, **{field: t})


def _x(shape, seed):
    g = torch.Generator()
    g.manual_seed(seed)
    return torch.randn(*shape, generator=g)


def _ln(x, w, b):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w, b)


def _double(w):
    vals = {f.name: getattr(w, f.name) for f in dataclasses.fields(w)}
    return type(w)(**{k: None if v is None else v.double().cpu() for k, v in vals.items()})


def assert_same_kind(got, want64, rtol, product=None):
    """NaN, infinities and their signs as in ``want64`` rounded to float32, the
    rest close. Where ``product``, the last value that float32 rounds before it
    (``want64`` itself), is within 1 % of the overflow line, either may come."""
    got, want = got.cpu().double(), want64.float()
    product = want64 if product is None else product
    edge = (product.abs() > 0.99 * FLT_MAX) & (product.abs() < 1.01 * FLT_MAX)
    nan, inf = torch.isnan(want) & ~edge, torch.isinf(want) & ~edge
    assert torch.equal(torch.isnan(got) & ~edge, nan)
    assert torch.equal(torch.where(inf, got, 0.0), torch.where(inf, want64.sign() * INF, 0.0))
    fin = ~(nan | inf | edge)
    size = torch.where(fin, want64, 0.0).abs().flatten(0, -2).amax(0) + 1.0  # per output channel
    err = (torch.where(fin, got - want64, 0.0).abs() / size).max()
    assert float(err) <= rtol, float(err)


@pytest.mark.parametrize("field,value", [("g_out_weight", INF), ("g_out_weight", -INF), ("g_out_weight", ROUNDS_UP),
                                         ("p_out_weight", INF), ("p_out_weight", FLT_MAX),
                                         ("p_out_weight", -ROUNDS_UP), ("g_in_weight", -INF),
                                         ("norm_out_bias", INF), ("norm_out_bias", -ROUNDS_UP),
                                         ("norm_in_weight", 1e37)])
@pytest.mark.parametrize("n", [20, 70])
def test_trimul_fp32(field, value, n):
    say(f"nonfinite trimul fp32 {field}={value} n={n}")
    w = P.pack_trimul_torch(P.trimul_to_protenix(syn.trimul_weights(seed=3)), torch.float32, "cuda")
    w = _set(w, field, 77 if "norm" in field else (5, 77), value)
    if field == "norm_in_weight":  # for the output gate alone: a b past float32's range is NaN after its LayerNorm
        w = _set(_set(w, "p_in_weight", (slice(None), 77), 0.0), "g_in_weight", (slice(None), 77), 0.0)
    x = _x((1, n, n, 128), 1)
    got = kernels.trimul(x.cuda(), None, w, "outgoing")
    torch.cuda.synchronize()
    d = _double(w)
    xn = _ln(x[0].double(), d.norm_in_weight, d.norm_in_bias)
    ab = torch.sigmoid(xn @ d.g_in_weight.T) * (xn @ d.p_in_weight.T)
    o = torch.einsum("ikc,jkc->ijc", ab[..., :128], ab[..., 128:])
    p = _ln(o, d.norm_out_weight, d.norm_out_bias) @ d.p_out_weight.T
    want = p.float().double() * torch.sigmoid(xn @ d.g_out_weight.T)
    # 1e-4: the float32 bar of every check, at results of order one
    assert_same_kind(got[0], want, 1e-4, p)


@pytest.mark.parametrize("field,value", [("g_weight", INF), ("g_weight", -ROUNDS_UP), ("o_weight", -INF),
                                         ("o_weight", FLT_MAX)])
def test_triattn_fp32(field, value):
    n = 20
    say(f"nonfinite triattn fp32 {field}={value}")
    w = P.pack_triattn_protenix(P.triattn_to_protenix(syn.triattn_weights(seed=4)), torch.float32, "cuda")
    w = _set(w, field, (5, 77), value)
    x = _x((1, n, n, 128), 2)
    got = kernels.triattn(x.cuda(), None, w)
    torch.cuda.synchronize()
    d = _double(w)
    xn = _ln(x[0].double(), d.norm_weight, d.norm_bias)
    split = lambda t: t.reshape(n, n, 4, 32).permute(0, 2, 1, 3)  # noqa: E731
    q, k, v = (split(xn @ t.T) for t in (d.q_weight, d.k_weight, d.v_weight))
    s = q @ k.transpose(-1, -2) * 32 ** -0.5 + (xn @ d.bias_weight.T).permute(2, 0, 1)
    o = (torch.softmax(s, -1) @ v).permute(0, 2, 1, 3).reshape(n, n, 128)
    want = (o * torch.sigmoid(xn @ d.g_weight.T)) @ d.o_weight.T
    assert_same_kind(got[0], want, 1e-4)


@pytest.mark.parametrize("scale", [1e25, 1e18])
@pytest.mark.parametrize("field,value", [(None, None), ("w_o", INF), ("w_o", ROUNDS_UP), ("w_b", -INF)])
def test_transition_fp32(field, value, scale):
    """At 1e25 the gated hidden unit 9 overflows float32 (or is -0), at 1e18 it
    stays finite."""
    rows = 70
    say(f"nonfinite transition fp32 {field}={value} scale={scale}")
    w = P.pack_transition_torch(P.transition_to_protenix(syn.transition_weights(seed=5)), torch.float32, "cuda")
    w = _set(w, "w_a", 9, w.w_a[9] * scale)
    w = _set(w, "w_b", 9, w.w_b[9] * scale)
    if field is not None:
        w = _set(w, field, (17, 33), value)
    x = _x((rows, 128), 3)
    got = kernels.transition(x.cuda(), w)
    torch.cuda.synchronize()
    d = _double(w)
    xn = _ln(x.double(), d.norm_weight, d.norm_bias)
    a, b = xn @ d.w_a.T, xn @ d.w_b.T
    h = (a * torch.sigmoid(a)).float() * b.float()  # float32's own overflow
    want = h.double() @ d.w_o.T
    assert_same_kind(got, want, 1e-4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,n", [(5, 40), (9, 100), (81, 430), (81, 500), (1, 70)])
@pytest.mark.parametrize("where", ["q", "bias"])
def test_core_nan_of_one_query(where, rows, n, dtype):
    """64- and 128-query workgroups, padded lengths that are even and odd
    multiples of 64, the single-row pass and the float32 one."""
    say(f"core NaN in {where} rows={rows} n={n} {dtype}")
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    q, k, v = (torch.randn(1, rows, 4, n, 32, generator=g, device="cuda").to(dtype) for _ in range(3))
    tb = torch.randn(1, 1, 4, n, n, generator=g, device="cuda").to(dtype)
    clean = kernels.triattn_core(q, k, v, tb, None, scale=32 ** -0.5)
    row, head, j = rows // 2, 2, n // 2 + 3
    bad = torch.zeros(1, rows, 4, n, dtype=torch.bool, device="cuda")
    if where == "q":
        q[0, row, head, j, 7] = math.nan
        bad[0, row, head, j] = True
    else:
        tb[0, 0, head, j, 5] = math.nan
        bad[0, :, head, j] = True
    got = kernels.triattn_core(q, k, v, tb, None, scale=32 ** -0.5)
    torch.cuda.synchronize()
    assert torch.equal(torch.isnan(got).all(-1), bad) and torch.equal(torch.isnan(got).any(-1), bad)
    # the rest: recomputed with another softmax offset at most (bf16: 2^-8 a
    # rounding of the probabilities and of the output)
    diff = torch.where(bad[..., None], 0.0, (got - clean).float()).abs().max()
    assert float(diff) <= (3e-2 if dtype == torch.bfloat16 else 1e-5) * float(clean.float().abs().max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("c_z,c_h", [(128, 128), (64, 128), (96, 128), (384, 384), (264, 72)])
@pytest.mark.parametrize("n", [37, 70, 200])
def test_trimul_padding_is_zero(n, c_z, c_h, dtype):
    """The operands' rows are padded past n. The LayerNorm of the padding's zero
    rows is NaN at eps = 0, and an infinite gate weight times a zero LayerNorm
    bias is too; neither may reach the contraction."""
    say(f"trimul padding n={n} {c_z} {c_h} {dtype}")
    w = P.pack_trimul_torch(P.trimul_to_protenix(syn.trimul_weights(c_z, c_h, seed=3)), dtype, "cuda")
    x = _x((1, n, n, c_z), 4).cuda().to(dtype)
    for direction in ("outgoing", "incoming"):
        got = kernels.trimul(x, None, w, direction, eps=0.0)
        want = kernels.trimul(x, None, w, direction, eps=1e-30)  # the same LayerNorms on rows that vary
        torch.cuda.synchronize()
        assert torch.isfinite(want).all() and torch.equal(got, want)
    inf = dataclasses.replace(_set(w, "g_in_weight", (5, 17), INF), norm_in_bias=torch.zeros_like(w.norm_in_bias))
    got = kernels.trimul(x, None, inf, "outgoing")
    torch.cuda.synchronize()
    assert torch.isfinite(got).all()
