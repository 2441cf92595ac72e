"""Register tiles whose last round of workgroups is cut into smaller tiles: every result there, whatever part of a tile lies past the rows or columns."""
import numpy as np
import pytest

import fastnn_amd
from fastnn_amd import lib as flib
from gpu_common import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [flib.DT_I8, flib.DT_I4, flib.DT_U4])
@pytest.mark.parametrize("waves,tail,m,k,n", [(1, 2, 1090, 300, 3900), (1, 4, 1090, 300, 3900), (1, 4, 1040, 200, 4000), (1, 2, 200, 64, 17000), (2, 4, 530, 1000, 3900),
                                              (2, 4, 514, 130, 4096), (1, 4, 1024, 64, 4096)])
def test_the_last_round(dt, waves, tail, m, k, n):
    """Sums of the same integers, so the bound of every f32-activation MatMul, 2e-5 of the largest result; the whole rounds are the bits of tiles that are not cut."""
    rng = np.random.default_rng(m + n + dt)
    pw = fastnn_amd.quantize_weights(dt, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[m - 1, k - 1] = np.inf
    bias = (rng.standard_normal(n) * 0.1).astype(np.float32)
    with fastnn_amd.HipContext(0) as ctx:
        h = ctx.register(pw)
        want = a[:-1].astype(np.float64) @ ctx.dequant(h, n, k).T.astype(np.float64) + bias
        ctx.set_option(flib.OPT_FRAGMENT, 1 << 14 | tail << 3 | waves)
        got = ctx.qmatmul(h, a, n, bias=bias)
        ctx.set_option(flib.OPT_FRAGMENT, 1 << 14 | waves)
        plain = ctx.qmatmul(h, a, n, bias=bias)
        assert_close(got[:-1], want, 2e-5)
        assert not np.isfinite(got[-1]).any()
        same = (got[:-1] == plain[:-1]).mean()
        assert same > 0.75, same
        if k >= 300:                     # (K in several parts there: other roundings, so that the cut tiles have run)
            assert same < 1
        ctx.release(h)
