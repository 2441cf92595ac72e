"""The digit planes of the register tiles' operand (four values a thread and pass) against the oracle: rows that stay in registers and rows
that are read twice, rows that end anywhere, rows that are not numbers."""
import numpy as np
import pytest

import fastnn_amd
from fastnn_amd import lib as flib
from gpu_common import assert_close, to_oracle

pytestmark = pytest.mark.gpu
WAVE = 1 << 14   # FNN_OPT_FRAGMENT: the register tiles


@pytest.mark.parametrize("dt", [flib.DT_I8, flib.DT_I4, flib.DT_U4])
@pytest.mark.parametrize("k", [130, 2047, 2052, 8191, 8193, 12002])
def test_against_the_oracle(orc, dt, k):
    """2e-5 of the largest result, as for every f32-activation MatMul."""
    rng = np.random.default_rng(k + dt)
    m, n = 35, 140
    pw = fastnn_amd.quantize_weights(dt, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::61] *= 100.0
    a[3] = 0.0
    want = orc.qmatmul(to_oracle(orc, pw), a, order=2)
    with fastnn_amd.HipContext(0) as ctx:
        h = ctx.register(pw)
        ctx.set_option(flib.OPT_FRAGMENT, WAVE | 2)
        assert_close(ctx.qmatmul(h, a, n), want, 2e-5)
        # a value that is no finite number makes its row's results no numbers, and no other row's
        bad = a.copy()
        bad[5, k - 1] = np.inf
        bad[9, 0] = np.nan
        bad[34, k // 2] = -np.inf
        got = ctx.qmatmul(h, bad, n)
        rows = [5, 9, 34]
        assert np.isnan(got[rows]).all()
        keep = [r for r in range(m) if r not in rows]
        assert_close(got[keep], want[keep], 2e-5)
        ctx.release(h)
