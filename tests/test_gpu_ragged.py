"""Pair lengths that are no multiple of any tile, bf16 tri-mul and tri-attn.

The padding rule gives an exact check: a tail of masked tokens contributes
zeros to the contraction, every position's own arithmetic is unchanged, and
both contraction tile sizes accumulate in the same order, so the n x n corner
of an N x N call whose last N - n tokens are masked is bit-identical to the
n x n call. The lengths sit around the edges of the 64-column rows, the
128- and 256-wide tiles and the rule that picks between those. The padded
side is checked against the oracle in test_gpu_triangle.py. The same holds
for tri-attn (masked keys have probability zero, key blocks accumulate in one
order), around the edges of the 64-key blocks, of the 64- and 128-query tiles
and of the rule between those.
"""

from __future__ import annotations

import pytest
import torch

from foldjax_amd import _lib, kernels
from foldjax_amd import params as P
from foldjax_amd import synthetic as syn
from tests.gpu_util import say

pytestmark = pytest.mark.gpu


def _weights(dtype, c_z=128, seed=5):
    return P.pack_trimul_torch(P.trimul_to_protenix(syn.trimul_weights(c_z, 128, seed=seed)), dtype, "cuda")


def _pair(n, dtype, c_z=128, seed=1):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(1, n, n, c_z, generator=g, device="cuda").to(dtype)


@pytest.mark.parametrize("n,padded", [(1, 64), (37, 64), (63, 128), (65, 256), (127, 128), (129, 256), (255, 320),
                                      (257, 320), (383, 512), (385, 512), (511, 577), (591, 640)])
@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
def test_trimul_corner_of_a_masked_call(n, padded, direction):
    say(f"ragged trimul n={n} in {padded} {direction}")
    w = _weights(torch.bfloat16)
    z = _pair(padded, torch.bfloat16)
    tok = (torch.arange(padded, device="cuda") < n).to(torch.bfloat16)
    want = kernels.trimul(z, torch.outer(tok, tok)[None], w, direction, residual=z)[:, :n, :n]
    zn = z[:, :n, :n].contiguous()
    got = kernels.trimul(zn, None, w, direction, residual=zn)
    torch.cuda.synchronize()
    assert torch.isfinite(got.float()).all()
    assert torch.equal(got, want)


def test_trimul_without_row_padding():
    """The static scratch does not hold three 341-token items with padded
    rows: the call runs on unpadded rows and gives the same bits."""
    n, batch = 341, 3
    say(f"trimul unpadded rows n={n} batch={batch}")
    lib = _lib.load()
    assert lib.fjx_trimul_workspace_size(batch, n, 128, 128, _lib.FJX_DTYPE_BF16) > _lib.NOALLOC_SCRATCH_BYTES
    w = _weights(torch.bfloat16)
    z = torch.cat([_pair(n, torch.bfloat16, seed=s) for s in range(batch)])
    want = kernels.trimul(z, None, w, "incoming")
    got = kernels.trimul(z, None, w, "incoming", no_alloc=True)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("n,padded", [(2, 64), (37, 64), (64, 128), (65, 192), (129, 192), (150, 256), (170, 256),
                                      (191, 384), (257, 320), (300, 512), (449, 577)])
@pytest.mark.parametrize("starting", [True, False])
def test_triattn_corner_of_a_masked_call(n, padded, starting):
    say(f"ragged triattn n={n} in {padded} starting={starting}")
    w = P.pack_triattn_protenix(P.triattn_to_protenix(syn.triattn_weights(seed=6)), torch.bfloat16, "cuda")
    z = _pair(padded, torch.bfloat16)
    tok = (torch.arange(padded, device="cuda") < n).to(torch.bfloat16)
    want = kernels.triattn(z, torch.outer(tok, tok)[None], w, starting=starting, residual=z)[:, :n, :n]
    zn = z[:, :n, :n].contiguous()
    got = kernels.triattn(zn, None, w, starting=starting, residual=zn)
    torch.cuda.synchronize()
    assert torch.isfinite(got.float()).all()
    assert torch.equal(got, want)


@pytest.mark.parametrize("mul", [1.0, 40.0])
@pytest.mark.parametrize("rows,n", [(1, 100), (5, 1), (5, 40), (3, 100), (9, 150), (81, 300), (81, 330)])
def test_triattn_core_at_every_tile(rows, n, mul):
    """The core reads q and k unpadded. At mul = 40, scores of hundreds in
    log2 units send workgroups of both query tiles, of odd and even block
    counts and of the half-empty last tile to the offset kernel. The reference is float32 torch on the same bf16 values; the
    kernel's bf16 probabilities and output leave at most 2^-8 of the largest
    value each (2^-9 per rounding, sums of positive terms), 2e-2 as for every
    bf16 check."""
    say(f"triattn core rows={rows} n={n} mul={mul}")
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    q, k, v = (torch.randn(1, rows, 4, n, 32, generator=g, device="cuda").bfloat16() for _ in range(3))
    q = (q.float() * mul).bfloat16()
    tb = torch.randn(1, 1, 4, n, n, generator=g, device="cuda").bfloat16()
    keep = torch.rand(1, rows, n, generator=g, device="cuda") > 0.2
    keep[..., 0] = True
    mb = torch.where(keep, 0.0, -1e9)[:, :, None, None, :]
    got = kernels.triattn_core(q, k, v, tb, mb, scale=32 ** -0.5)
    # the kernels take scale * log2(e) into q in bf16
    log2e = 1.4426950408889634
    qs = (q.float() * (32 ** -0.5 * log2e)).bfloat16().float()
    s = (qs @ k.float().transpose(-1, -2).contiguous()) / log2e + tb.float() + mb
    want = torch.softmax(s, -1) @ v.float()
    torch.cuda.synchronize()
    assert torch.isfinite(got.float()).all()
    err = (got.float() - want).norm() / want.norm()
    assert err <= 2e-2, float(err)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,heads,c_s", [(1, 16, 384), (17, 3, 24), (65, 16, 384), (130, 20, 320), (200, 32, 160)])
def test_single_attention_head_widths(n, heads, c_s, dtype):
    """The pair bias past one 16-head tile and at lengths that are no multiple
    of 16, and the gated output of head widths 8, 24 and 5 and 16, against
    float64 torch on the same values."""
    say(f"single attention n={n} heads={heads} c_s={c_s} {dtype}")
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    lin = lambda o, i: (rnd(o, i) / i ** 0.5).to(dtype)  # noqa: E731
    w = kernels.SingleAttentionWeights(
        pre_norm_weight=(1 + 0.1 * rnd(c_s)).to(dtype), pre_norm_bias=(0.1 * rnd(c_s)).to(dtype),
        z_norm_weight=(1 + 0.1 * rnd(128)).to(dtype), z_norm_bias=(0.1 * rnd(128)).to(dtype), z_weight=lin(heads, 128),
        q_weight=lin(c_s, c_s), q_bias=(0.1 * rnd(c_s)).to(dtype), k_weight=lin(c_s, c_s), v_weight=lin(c_s, c_s),
        g_weight=lin(c_s, c_s), o_weight=lin(c_s, c_s)).to(dtype, "cuda")
    s, z = rnd(1, n, c_s).to(dtype), rnd(1, n, n, 128).bfloat16()
    mask = (torch.arange(n, device="cuda") < max(1, n - 3)).to(dtype)[None]
    got = kernels.single_attention(s, z, mask, w)
    ln = lambda x, a, b: torch.nn.functional.layer_norm(x.double(), x.shape[-1:], a.double(), b.double())  # noqa: E731
    mm = lambda x, m: x @ m.double().t().contiguous()  # noqa: E731
    x = ln(s[0], w.pre_norm_weight, w.pre_norm_bias)
    split = lambda t: t.reshape(n, heads, -1).permute(1, 0, 2).contiguous()  # noqa: E731
    q, k, v = split(mm(x, w.q_weight) + w.q_bias.double()), split(mm(x, w.k_weight)), split(mm(x, w.v_weight))
    sc = q @ k.transpose(1, 2).contiguous() * (c_s // heads) ** -0.5
    sc = sc + mm(ln(z[0], w.z_norm_weight, w.z_norm_bias), w.z_weight).permute(2, 0, 1) + 1e6 * (mask[0].double() - 1)
    o = (torch.softmax(sc, -1) @ v).permute(1, 0, 2).reshape(n, c_s)
    want = mm(o * torch.sigmoid(mm(x, w.g_weight)), w.o_weight)
    torch.cuda.synchronize()
    err = float((got[0].double() - want).norm() / want.norm())
    assert err <= (2e-5 if dtype == torch.float32 else 2e-2), err


@pytest.mark.parametrize("n,padded", [(1, 64), (63, 128), (65, 192), (127, 192), (129, 200)])
@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
def test_trimul_fp32_corner_of_a_masked_call(n, padded, direction):
    """As for bf16: the fp32 path's splits, its 64-position tiles and its
    128-wide contraction tiles leave every valid position's arithmetic alone."""
    say(f"ragged fp32 trimul n={n} in {padded} {direction}")
    w = _weights(torch.float32)
    z = _pair(padded, torch.float32)
    tok = (torch.arange(padded, device="cuda") < n).float()
    want = kernels.trimul(z, torch.outer(tok, tok)[None], w, direction, residual=z)[:, :n, :n]
    zn = z[:, :n, :n].contiguous()
    got = kernels.trimul(zn, None, w, direction, residual=zn)
    torch.cuda.synchronize()
    assert torch.isfinite(got).all()
    assert torch.equal(got, want)


@pytest.mark.parametrize("n,batch", [(400, 1), (418, 1), (133, 9), (1, 3000), (65, 40)])
def test_trimul_fp32_noalloc_bits(n, batch):
    """The static scratch holds the split planes up to its largest float32
    length, and of larger batches as many items as fit at a time: the bits of
    the call with a workspace. (65, 40): 22 and 18 items; (1, 3000): 2926."""
    say(f"trimul fp32 noalloc n={n} batch={batch}")
    w = _weights(torch.float32)
    z = torch.cat([_pair(n, torch.float32, seed=s % 7) for s in range(batch)])
    mask = (torch.rand(batch, n, n, device="cuda") > 0.2).float()
    out_mask = (torch.rand(batch, n, n, device="cuda") > 0.1).float()
    want = kernels.trimul(z, mask, w, "incoming", residual=z, out_mask=out_mask)
    got = kernels.trimul(z, mask, w, "incoming", residual=z, out_mask=out_mask, no_alloc=True)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("n", [1, 5, 8, 33])
@pytest.mark.parametrize("heads", [1, 16])
def test_transition_fp32_with_pair_bias(n, heads):
    """The fp32 pair transition at row counts around its 64-row tile, with every
    option and the pair bias, against float64 torch (fp32 products: 1e-5)."""
    say(f"transition fp32 n={n} heads={heads}")
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    w = P.pack_transition_torch(P.transition_to_protenix(syn.transition_weights(seed=3)), torch.float32, "cuda")
    aw = kernels.SingleAttentionWeights(
        pre_norm_weight=None, pre_norm_bias=None, z_norm_weight=1 + 0.1 * rnd(128), z_norm_bias=0.1 * rnd(128),
        z_weight=rnd(heads, 128), q_weight=rnd(32, 32), q_bias=None, k_weight=rnd(32, 32), v_weight=rnd(32, 32),
        g_weight=rnd(32, 32), o_weight=rnd(32, 32))
    x, res = rnd(2, n, n, 128), rnd(2, n, n, 128)
    rm, om = (rnd(2, n, n) > 0).float() * 0.5, (rnd(2, n, n) > -1).float()
    out, pb = kernels.transition(x, w, row_mask=rm, residual=res, out_mask=om, pair_bias_for=aw)
    ln = lambda v, a, b: torch.nn.functional.layer_norm(v, (128,), a.double(), b.double())  # noqa: E731
    mm = lambda v, m: v @ m.double().t().contiguous()  # noqa: E731
    xn = ln(x.double(), w.norm_weight, w.norm_bias)
    y = mm(torch.nn.functional.silu(mm(xn, w.w_a)) * mm(xn, w.w_b), w.w_o) * rm[..., None] + res
    y = y * (om != 0)[..., None]
    bias = mm(ln(out.double(), aw.z_norm_weight, aw.z_norm_bias), aw.z_weight).permute(0, 3, 1, 2) * 1.4426950408889634
    torch.cuda.synchronize()
    assert float((out.double() - y).norm() / y.norm()) <= 1e-5
    assert float((pb[:, :, :n, :n].double() - bias).norm() / bias.norm()) <= 1e-5
    assert not pb[:, :, n:].any() and not pb[..., n:].any()


@pytest.mark.parametrize("c,bias", [(128, torch.float32), (128, torch.bfloat16), (128, None), (64, None), (96, None)])
@pytest.mark.parametrize("n", [1, 5, 90, 91, 128, 150])
def test_transition_rows_do_not_depend_on_the_tile(n, c, bias):
    """A row's arithmetic is its own, so one item alone (32- and 64-row tiles at
    these lengths) has the bits it has among enough items for 128-row tiles."""
    say(f"transition tiles n={n} c={c} bias={bias}")
    dtype = torch.bfloat16
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    batch = 33000 // (n * n) + 2
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)  # noqa: E731
    w = P.pack_transition_torch(P.transition_to_protenix(syn.transition_weights(c, seed=3)), dtype, "cuda")
    x, res = rnd(batch, n, n, c), rnd(batch, n, n, c)
    rm, om = (rnd(batch, n, n) > 0).to(dtype) * 0.5, (rnd(batch, n, n) > -1).to(dtype)
    aw = None
    if bias is not None:
        aw = kernels.SingleAttentionWeights(
            pre_norm_weight=None, pre_norm_bias=None, z_norm_weight=1 + 0.1 * rnd(c), z_norm_bias=0.1 * rnd(c),
            z_weight=rnd(16, c), q_weight=rnd(64, 64), q_bias=None, k_weight=rnd(64, 64), v_weight=rnd(64, 64),
            g_weight=rnd(64, 64), o_weight=rnd(64, 64)).to(bias, "cuda")
    want = kernels.transition(x, w, row_mask=rm, residual=res, out_mask=om, pair_bias_for=aw)
    one = [t[1:2].contiguous() for t in (x, res, rm, om)]
    got = kernels.transition(one[0], w, row_mask=one[2], residual=one[1], out_mask=one[3], pair_bias_for=aw)
    torch.cuda.synchronize()
    if aw is not None:
        (want, want_pb), (got, got_pb) = want, got
        assert torch.equal(getattr(got_pb, "bias", got_pb)[0], getattr(want_pb, "bias", want_pb)[1])
    assert torch.isfinite(got.float()).all()
    assert torch.equal(got[0], want[1])


def test_triattn_core_of_very_many_rows():
    """65 items of 65535 one-token rows and 4 heads: 17 million head rows, more
    blocks than one launch takes. One key has probability one: the output is v."""
    batch, rows = 65, 65535
    say(f"triattn core batch={batch} rows={rows}")
    v = torch.randn(batch, rows, 4, 1, 32, device="cuda", dtype=torch.bfloat16)
    tb = torch.zeros(batch, 1, 4, 1, 1, device="cuda", dtype=torch.bfloat16)
    got = kernels.triattn_core(v, v, v, tb, None, scale=0.05)
    torch.cuda.synchronize()
    assert torch.equal(got, v)
    del got, v
    torch.cuda.empty_cache()  # 70 GB of workspace
