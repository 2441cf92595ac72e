"""The host weight packers at the edges of their panels of 32 channels, from [N, K] and from [K, N] matrices, against the
oracle bit for bit."""
import numpy as np
import pytest

import fastnn_amd
from fastnn_amd import lib as flib


@pytest.mark.parametrize("dt", range(8))
@pytest.mark.parametrize("rows,inner", [(1, 1), (31, 15), (32, 64), (33, 129), (97, 1003), (300, 1024)])
@pytest.mark.parametrize("kind", ["normal", "special", "ties"])
def test_packers_at_panel_edges(orc, dt, rows, inner, kind):
    rng = np.random.default_rng(rows * 7 + inner)
    w = (rng.standard_normal((rows, inner)) * 0.02).astype(np.float32)
    if kind == "ties":          # values on and around the rounding boundaries, signed zeros
        w = (rng.integers(-9, 9, (rows, inner)) / 2).astype(np.float32)
        w[:, ::3] = -0.0
    if kind == "special":
        w[0] = 0.5
        w[-1] = 1e-38
        if dt != flib.DT_I4CB:  # (the codebook packer refuses NaN)
            w[rng.random(w.shape) < 0.02] = np.inf
            w[rng.random(w.shape) < 0.02] = np.nan
    po = orc.quantize(dt, w)
    for pw in (fastnn_amd.quantize_weights(dt, w), fastnn_amd.quantize_weights_kn(dt, np.ascontiguousarray(w.T))):
        assert np.array_equal(pw.words, po.words)
        assert np.array_equal(pw.scales, po.scales, equal_nan=True) and np.array_equal(pw.zeros, po.zeros, equal_nan=True)
        if dt == flib.DT_I4CB:
            assert pw.codebook.tobytes() == po.codebook.tobytes()
