"""fjx_trimul_fwd on a workspace without room for padded rows or planes: what
the call needed before either, and still accepts."""

from __future__ import annotations

import ctypes

import pytest
import torch

from foldjax_amd import _lib, kernels
from foldjax_amd import params as P
from foldjax_amd import synthetic as syn
from tests.gpu_util import say

pytestmark = pytest.mark.gpu


def _up(nbytes):
    return (nbytes + 255) // 256 * 256


def unpadded_bytes(batch, n, c_z, c_h, es):
    """a, b and o on rows of n elements; at general widths also LN(x), the gated
    product, the output gate and the two input weights interleaved."""
    pos = batch * n * n * es
    if c_h == 128 and c_z in (32, 64, 96, 128):
        return 3 * _up(pos * 128)
    return 3 * _up(pos * c_h) + 2 * _up(pos * c_z) + _up(2 * pos * c_h) + _up(4 * c_h * c_z * es)


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("batch,n,c_z,c_h", [(1, 37, 128, 128), (3, 100, 128, 128), (1, 256, 128, 128),
                                             (2, 65, 64, 128), (2, 33, 384, 384), (1, 100, 128, 64)])
def test_trimul_on_an_unpadded_workspace(batch, n, c_z, c_h, dtype, direction):
    say(f"trimul unpadded workspace batch={batch} n={n} {c_z} {c_h} {dtype} {direction}")
    lib = _lib.load()
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    x = torch.randn(batch, n, n, c_z, generator=g, device="cuda").to(dtype)
    mask = (torch.rand(batch, n, n, generator=g, device="cuda") > 0.2).to(dtype)
    w = P.pack_trimul_torch(P.trimul_to_protenix(syn.trimul_weights(c_z, c_h, seed=5)), dtype, "cuda")
    want = kernels.trimul(x, mask, w, direction, residual=x)
    code = _lib.FJX_DTYPE_BF16 if dtype == torch.bfloat16 else _lib.FJX_DTYPE_F32
    size = unpadded_bytes(batch, n, c_z, c_h, x.element_size())
    buf = torch.full((size + 4096,), 0xFF, dtype=torch.uint8, device="cuda")  # NaN in both dtypes
    out = torch.empty_like(x)
    a = _lib.TriMulArgs(
        batch=batch, n=n, c_z=c_z, c_h=c_h,
        direction=_lib.FJX_OUTGOING if direction == "outgoing" else _lib.FJX_INCOMING, dtype=code, eps=1e-5,
        x=x.data_ptr(), mask=mask.data_ptr(), residual=x.data_ptr(), out=out.data_ptr(), workspace=buf.data_ptr(),
        workspace_bytes=size, **{k: getattr(w, k).data_ptr() for k in (
            "norm_in_weight", "norm_in_bias", "p_in_weight", "g_in_weight", "norm_out_weight", "norm_out_bias",
            "p_out_weight", "g_out_weight")})
    _lib.check(lib.fjx_trimul_fwd(ctypes.byref(a), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert bool((buf[size:] == 0xFF).all()), "written past the workspace's end"
    # the fused bf16 kernels compute the same bits on either layout; at general
    # widths the unpadded route rounds the gated product once, the other its two
    # factors and the product: at most 2^-9 a rounding in a, b and, past the
    # LayerNorm, the output, 4 x 2^-9 in all; float32's two paths each stay
    # within a few units of float32's roundoff
    err = float((out.float() - want.float()).norm() / want.float().norm())
    if dtype == torch.bfloat16 and c_h == 128:
        assert torch.equal(out, want)
    else:
        assert err <= (4 * 2 ** -9 if dtype == torch.bfloat16 else 2e-6), err
    if c_h == 128:  # less is refused on the host
        a.workspace_bytes = size - 1
        assert lib.fjx_trimul_fwd(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == _lib.FJX_ERR_WORKSPACE


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("c_z,c_h", [(128, 128), (64, 128), (96, 128), (384, 384), (264, 72), (128, 576)])
@pytest.mark.parametrize("n", [1, 37, 70])
def test_trimul_leaves_nothing_to_the_workspace(n, c_z, c_h, dtype, monkeypatch):
    """Every byte that a call reads of its workspace it has written: NaN left
    there changes nothing."""
    say(f"trimul workspace contents n={n} {c_z} {c_h} {dtype}")
    x = torch.randn(1, n, n, c_z, device="cuda").to(dtype)
    w = P.pack_trimul_torch(P.trimul_to_protenix(syn.trimul_weights(c_z, c_h, seed=5)), dtype, "cuda")
    empty = torch.empty

    def filled(value):
        def make(*shape, **kw):
            t = empty(*shape, **kw)
            return t.fill_(value) if kw.get("dtype") is torch.uint8 else t
        return make

    out = []
    for value in (0, 0xFF):
        monkeypatch.setattr(torch, "empty", filled(value))
        out.append(kernels.trimul(x, None, w, "outgoing"))
        torch.cuda.synchronize()
    assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_trimul_where_the_full_workspace_does_not_fit(dtype, monkeypatch):
    n = 70
    say(f"trimul out of memory {dtype}")
    x = torch.randn(2, n, n, 128, device="cuda").to(dtype)
    w = P.pack_trimul_torch(P.trimul_to_protenix(syn.trimul_weights(seed=5)), dtype, "cuda")
    want = kernels.trimul(x, None, w, "outgoing")
    limit, empty, asked = unpadded_bytes(2, n, 128, 128, x.element_size()), torch.empty, []

    def scarce(*shape, **kw):
        if kw.get("dtype") is torch.uint8:
            asked.append(shape[0])
            if shape[0] > limit:
                raise torch.OutOfMemoryError("no room")
        return empty(*shape, **kw)

    monkeypatch.setattr(torch, "empty", scarce)
    got = kernels.trimul(x, None, w, "outgoing")
    torch.cuda.synchronize()
    assert len(asked) == 2 and asked[1] == limit
    assert float((got.float() - want.float()).norm() / want.float().norm()) <= 2e-6
