"""A reset clears every accumulation buffer to its last pixel."""
import numpy as np
import pytest

from ohao_engine_amd import denoise as D
from ohao_engine_amd import ohpt
from ohao_engine_amd import scenes as S

pytestmark = pytest.mark.gpu


def buffers(ctx):
    albedo, normal, depth = ctx.read_aovs()      # the albedo's alpha reads as 1
    return (*ctx.read_moments(), ctx.read_display_sums(), albedo[..., :3], normal, depth)


@pytest.mark.parametrize("W,H", [(1, 1), (51, 5), (16, 16), (257, 3)])
def test_reset_clears_all_buffers(W, H):
    sc = S.cornell_box(W, H)
    ctx = ohpt.Context(W, H)
    ctx.load_scene(sc)
    D.with_guides(ctx, sc.settings)
    ctx.render(3)
    assert all(np.abs(a).max() > 0 for a in buffers(ctx))
    ctx.reset()
    assert all(np.all(a == 0.0) for a in buffers(ctx))
    ctx.close()
