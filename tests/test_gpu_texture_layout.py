"""Texels move between the caller's layout and the packed one on the device: every
channel count, host and device sources, sizes below one block, around the mean's
grid (512 blocks of 256 texels) and with a remainder. The host and the device route
are compared with each other, and their results with the CPU oracle and with the same
frames of textures that numpy has padded to four channels."""
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
    """The emitter table divides by the mean: a frame lit by an emissive texture must
    not depend on whether the texels came at the upload or later."""
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


def padded(a):
    """The four channels that a texture of fewer stands for: grey, two and zero, alpha one."""
    h, w, c = a.shape
    if c == 1:
        return np.repeat(a, 4, 2)
    out = np.zeros((h, w, 4), np.float32)
    out[..., :c] = a
    if c == 3:
        out[..., 3] = 1.0
    return out


@pytest.mark.parametrize("w,h", [(17, 3), (64, 64), (241, 17), (257, 513)])   # up to 4096 texels packed on the host
@pytest.mark.parametrize("channels", [1, 2, 3, 4])
def test_packed_texels_are_the_callers(oracle, w, h, channels):
    rng = np.random.default_rng(w + channels)
    a, b = (rng.random((h, w, channels), dtype=np.float32) for _ in range(2))
    base = S.lantern(freq=4, tex_size=8, texture=np.full((8, 8, 3), 0.5, np.float32))
    at = lambda t: S.Scene(**{**base.__dict__, "textures": [t], "width": 48, "height": 32})
    ctx = ohpt.Context(48, 32)
    ctx.load_scene(at(a))
    for tex in (a, b):
        o = oracle.OracleScene(at(padded(tex)))
        got = frame(ctx, tex, True)[..., :3]
        want, _ = o.render(1, base.settings.seed, precision=32)
        # the same arithmetic in FP32 but for the math library's functions; a channel in
        # another's place or another fill differs by more than a tenth
        assert np.abs(got - want).sum() < 1e-3 * np.abs(want).sum()
        assert np.array_equal(got, padded_frame(at(padded(tex))))
    ctx.close()


def padded_frame(sc):
    ctx = ohpt.Context(sc.width, sc.height)
    ctx.load_scene(sc)
    ctx.render(1)
    out = ctx.read_accum()[..., :3]
    ctx.close()
    return out


@pytest.mark.parametrize("channels", [1, 2, 3])
def test_unpacked_gradients_are_the_four_channel_ones(channels):
    """Sums in a fixed order: the channels that a texture has get the gradient that the same
    channels of its four-channel form get, bit for bit; a grey texel gets the sum of three."""
    rng = np.random.default_rng(channels + 9)
    tex = rng.random((37, 29, channels), dtype=np.float32) * 0.8 + 0.1
    base = S.lantern(freq=6, tex_size=8, texture=np.full((8, 8, 3), 0.5, np.float32))
    grads = []
    for t in (tex, padded(tex)):
        ctx = ohpt.Context(64, 48)
        ctx.load_scene(S.Scene(**{**base.__dict__, "textures": [t], "width": 64, "height": 48}))
        ctx.zero_gradients()
        ctx.adjoint(np.ones((48, 64, 4), np.float32), 2, deterministic=True)
        grads.append(ctx.texture_gradient(0, t.shape))
        ctx.close()
    got, four = grads
    assert np.abs(got).max() > 0
    if channels == 1:
        want = four[..., :3].astype(np.float64).sum(2)
        # three sums of the records against one of all of them: at most a few thousand FP32 additions
        assert np.abs(got[..., 0] - want).max() < 1e-4 * np.abs(four).max()
    else:
        assert np.array_equal(got, four[..., :channels])


@pytest.mark.parametrize("w,h", [(61, 30), (128, 64), (61, 139), (512, 256), (513, 256), (700, 411)])
@pytest.mark.parametrize("channels", [1, 2, 3, 4])
def test_mean_of_an_emissive_texture_chooses_between_two_emitters(oracle, w, h, channels):
    """The mean is half of the choice between the lamp and a textured emitter: with another
    mean than the caller's texels have, other paths go to the lamp than the oracle's."""
    rng = np.random.default_rng(w + channels)
    tex = rng.random((h, w, channels), dtype=np.float32) ** 2
    tex[h // 2:] *= 4.0                          # blocks of texels differ
    sc = S.cornell_box(48, 48)
    mats = sc.materials.copy()
    mats["emissive"][2] = 2.0                    # the right wall
    mats["emissive_tex"][2] = 0
    sc = S.Scene(**{**sc.__dict__, "textures": [tex], "materials": mats})
    o = oracle.OracleScene(S.Scene(**{**sc.__dict__, "textures": [padded(tex)]}))
    want, _ = o.render(4, sc.settings.seed, precision=32)
    for late in (False, True):
        ctx = ohpt.Context(48, 48)
        ctx.load_scene(S.Scene(**{**sc.__dict__, "textures": [np.ones_like(tex) if late else tex]}))
        if late:
            ctx.update_texture(0, torch.from_numpy(tex).cuda())
        ctx.reset()
        ctx.render(4)
        got = ctx.read_accum()[..., :3] * 4.0
        ctx.close()
        off = np.abs(got - want).sum() / np.abs(want).sum()
        assert off < 1e-3, off
