"""Environment tables are sums in column order, in FP32: in the middle row of an odd height the
sine of the latitude is exactly one, so numpy gives the row's table bit for bit, at widths around
the 2048 values that a block sums at once."""
import numpy as np
import pytest

from ohao_engine_amd import ohpt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [1, 5, 255, 257, 2047, 2048, 2049, 4099])
@pytest.mark.parametrize("H", [1, 3, 65])
def test_middle_row_is_the_sequential_sum(W, H):
    rng = np.random.default_rng(W + H)
    env = rng.random((H, W, 4), dtype=np.float32) ** 8 * 100
    ctx = ohpt.Context(16, 16)
    ctx.set_env(env)
    marg, cond, integral = ctx.export_env_cdf(W, H)
    ctx.close()
    f = np.float32
    p = env[H // 2]
    lum = (f(0.2126) * p[:, 0] + f(0.7152) * p[:, 1]) + f(0.0722) * p[:, 2]
    sums = np.add.accumulate(lum, dtype=np.float32)
    assert np.array_equal(cond[H // 2], sums / sums[-1])
    if H == 1:
        assert integral == sums[-1] and marg[0] == 1.0
    assert np.all(np.diff(marg) >= 0) and marg[-1] == 1.0
