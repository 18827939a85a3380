"""CPU check of the tri-mul workspace against what it must hold."""

from __future__ import annotations

import pytest

from foldjax_amd import _lib

F32, BF16 = _lib.FJX_DTYPE_F32, _lib.FJX_DTYPE_BF16


@pytest.mark.parametrize("n", [1, 7, 16, 33, 64, 100])
@pytest.mark.parametrize("c_z,c_h", [(264, 192), (384, 384), (128, 72)])
def test_float32_rows_are_padded_to_eight_elements(n, c_z, c_h):
    """Rows padded to 64 serve the LDS-DMA contraction, which float32 does not run
    at general widths: a, b and o take (n + 7) / 8 * 8 elements a row, and the other
    buffers (LN(x), the gated product, the gate) none past n."""
    batch = 100
    pitch = (n + 7) // 8 * 8
    size = _lib.load().fjx_trimul_workspace_size(batch, n, c_z, c_h, F32)
    want = 3 * batch * n * pitch * c_h * 4 + batch * n * n * (2 * c_z + 2 * c_h) * 4
    assert want <= size <= want + 8 * 256
