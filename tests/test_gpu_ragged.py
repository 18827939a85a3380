"""Pair lengths that are no multiple of any tile, bf16 tri-mul.

The padding rule gives an exact check: a tail of masked tokens contributes
zeros to the contraction, every position's own arithmetic is unchanged, and
both contraction tile sizes accumulate in the same order, so the n x n corner
of an N x N call whose last N - n tokens are masked is bit-identical to the
n x n call. The lengths sit around the edges of the 64-column rows, the
128- and 256-wide tiles and the rule that picks between those. The padded
side is checked against the oracle in test_gpu_triangle.py.
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
