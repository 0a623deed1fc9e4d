"""The fused pointwise pair with four and with eight waves per tile.

Launches of fewer than 400 32-pixel tiles use eight waves, larger ones four;
a row's sums run in the same order in both, so a row computed in a small call
equals the same row of a large call bit for bit.  Hidden and output widths with
fewer and more column tiles than waves, and rows not a multiple of a tile; the
values themselves are pinned against float64 by the small calls of
test_conv_kernels_gpu.py.
"""
import ctypes

import numpy as np
import pytest

from test_conv_kernels_gpu import _lib, _ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c,co,gated,residual", [(16, 16, False, True), (32, 32, True, True), (48, 96, False, False),
                                                 (64, 160, True, False), (64, 64, False, True)])
def test_small_and_large_calls_agree(c, co, gated, residual):
    lib = _lib()
    f, i = ctypes.POINTER(ctypes.c_float), ctypes.c_int
    lib.ppocr_probe_pointwise_pair.argtypes = [f, i, i, i, f, f, f, i, f, f, i, i, f]
    lib.ppocr_probe_pointwise_pair.restype = i
    rng = np.random.default_rng(c + co)
    m, hw, h2, few = 12 * 1100 + 7, 1100, 2 * c, 2 * 1100  # 413 tiles, 69 tiles
    x = rng.standard_normal((m, c)).astype(np.float32)
    gate = rng.uniform(0, 1, (-(-m // hw), c)).astype(np.float32) if gated else None
    w1 = (rng.standard_normal((h2, c)) / np.sqrt(c)).astype(np.float32)
    w2 = (rng.standard_normal((co, h2)) / np.sqrt(h2)).astype(np.float32)
    b1, b2 = (rng.standard_normal(n).astype(np.float32) for n in (h2, co))

    def run(first, rows):
        out = np.empty((rows, co), np.float32)
        part = np.ascontiguousarray(x[first:first + rows])
        g = None if gate is None else np.ascontiguousarray(gate[first // hw:])
        assert lib.ppocr_probe_pointwise_pair(_ptr(part), rows, hw, c, _ptr(g), _ptr(w1), _ptr(b1), h2, _ptr(w2),
                                              _ptr(b2), co, int(residual), _ptr(out)) == 0
        return out

    whole = run(0, m)
    assert np.isfinite(whole).all()
    for first in (0, 4 * hw, 10 * hw):
        rows = min(few + 7, m - first)
        assert np.array_equal(run(first, rows), whole[first:first + rows])
