"""Texels move between the caller's layout and the packed one on the device: every
channel count, host and device sources, sizes below one block, around the mean's
grid (512 blocks of 256 texels) and with a remainder."""
import numpy as np
import pytest
import torch

from ohao_engine_amd import ohpt
from ohao_engine_amd import scenes as S

pytestmark = pytest.mark.gpu


def frame(ctx, texture, device):
    """A directly lit floor filling the view, the texture as albedo."""
    t = torch.from_numpy(texture).cuda() if device else texture
    ctx.update_texture(0, t)
    ctx.reset()
    ctx.render(1)
    return ctx.read_accum()


@pytest.mark.parametrize("w,h", [(1, 1), (17, 3), (255, 1), (257, 513), (362, 363)])
@pytest.mark.parametrize("channels", [1, 2, 3, 4])
def test_upload_and_update_agree(w, h, channels):
    rng = np.random.default_rng(w * 1000 + channels)
    a = rng.random((h, w, channels), dtype=np.float32)
    b = rng.random((h, w, channels), dtype=np.float32)
    sc = S.lantern(freq=4, tex_size=8, texture=np.full((8, 8, 3), 0.5, np.float32))
    sc = S.Scene(**{**sc.__dict__, "textures": [a], "width": 48, "height": 32})
    ctx = ohpt.Context(48, 32)
    ctx.load_scene(sc)
    ctx.render(1)
    first = ctx.read_accum()
    other = frame(ctx, b, True)
    assert not np.array_equal(first, other) or w * h == 1
    assert np.array_equal(frame(ctx, b, False), other)
    assert np.array_equal(frame(ctx, a, True), first)
    ctx.close()


@pytest.mark.parametrize("channels", [1, 2, 3, 4])
def test_gradient_reads_agree(channels):
    rng = np.random.default_rng(channels)
    tex = rng.random((37, 29, channels), dtype=np.float32) * 0.8 + 0.1
    sc = S.lantern(freq=6, tex_size=8, texture=np.full((8, 8, 3), 0.5, np.float32))
    sc = S.Scene(**{**sc.__dict__, "textures": [tex], "width": 64, "height": 48})
    ctx = ohpt.Context(64, 48)
    ctx.load_scene(sc)
    ctx.zero_gradients()
    ctx.adjoint(np.ones((48, 64, 4), np.float32), 2, deterministic=True)
    host = ctx.texture_gradient(0, tex.shape)
    dev = torch.full(tex.shape, 7.0, device="cuda:0")
    ctx.texture_gradient_device(0, dev)
    assert np.array_equal(dev.cpu().numpy(), host) and np.abs(host).max() > 0
    ctx.close()


@pytest.mark.parametrize("channels", [1, 3, 4])
def test_mean_of_an_emissive_texture_weighs_its_triangles(channels):
    """The emitter table divides by the mean: a frame lit by an emissive texture of
    one value must not depend on whether the texels came at the upload or later."""
    rng = np.random.default_rng(channels)
    tex = rng.random((61, 130, channels), dtype=np.float32)
    frames = []
    for late in (False, True):
        sc = S.cornell_box(48, 48)
        ctx = ohpt.Context(48, 48)
        mats = sc.materials.copy()
        mats["emissive_tex"][mats["emissive"].max(axis=1) > 0] = 0
        sc = S.Scene(**{**sc.__dict__, "textures": [np.ones_like(tex) if late else tex], "materials": mats})
        ctx.load_scene(sc)
        if late:
            ctx.update_texture(0, torch.from_numpy(tex).cuda())
        ctx.reset()
        ctx.render(4)
        frames.append(ctx.read_accum())
        ctx.close()
    assert np.array_equal(frames[0], frames[1])
