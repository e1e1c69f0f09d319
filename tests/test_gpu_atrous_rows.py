"""Both forms of the a-trous iteration (one and four pixels per thread, the latter
from 400,000 pixels) against the oracle where a band of rows can go wrong: images
lower than a band of the largest step (64 rows), a last band with one row, one
column, widths around the 64-pixel blocks."""
import sys
from pathlib import Path

import numpy as np
import pytest

from ohao_engine_amd import denoise as D
from ohao_engine_amd import ohpt
from test_gpu_atrous import small_scene, sums_from_context

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "oracle"))
import atrous_ref  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(1, 1), (1, 131), (65, 2), (63, 65), (399999, 1),
                                 (12904, 31), (6250, 64), (6155, 65), (401, 998), (1, 400000)])
def test_row_bands_match_oracle(W, H):
    print(f"a-trous rows {W}x{H}", flush=True)
    sc = small_scene(64, 48)
    ctx = ohpt.Context(W, H)
    try:
        ctx.load_scene(sc)
        D.with_guides(ctx, sc.settings)
        ctx.set_render_seed(5)
        ctx.reset()
        ctx.render(2)
        out = ctx.denoise_atrous()
        ref = atrous_ref.denoise_atrous(*sums_from_context(ctx))
    finally:
        ctx.close()
    # FP32 against float64: an exponent of size e is off by a few 2^-24 e, and a tap of
    # weight exp(-e) e 2^-22 or less than 1e-6; display values are at most 1
    err = np.abs(out[..., :3] - ref[..., :3])
    assert np.all(np.isfinite(out)) and np.all(out[..., 3] == 1.0)
    assert err.max() <= 2e-4 and err.mean() < 1e-5
