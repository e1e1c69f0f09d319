"""What the library's host side leaves behind, watched without a GPU: the library runs in a
process of its own over tests/hip_recorder.cpp, which takes the HIP runtime's place, runs no
kernel, and counts copies that nothing has waited for and bytes that are allocated."""
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

PRELUDE = """
import ctypes as C, sys
sys.modules["torch"] = None                    # its own copy of the runtime stays out of this process
R = C.CDLL({recorder!r}, mode=C.RTLD_GLOBAL)   # found before the runtime that the library links
R.rec_allocated.restype = R.rec_peak.restype = C.c_size_t
R.rec_fail_malloc.argtypes = R.rec_fail_copy.argtypes = [C.c_long]
R.rec_launch.restype = C.c_char_p
sys.path.insert(0, {root!r})
import numpy as np
from ohao_engine_amd import ohpt, scenes as S

def launches():
    g = (C.c_uint32 * 3)()
    return [(R.rec_launch(i, g).decode(), tuple(g)) for i in range(R.rec_launches())]
"""


@pytest.fixture(scope="module")
def recorded(tmp_path_factory):
    lib = tmp_path_factory.mktemp("recorder") / "libhip_recorder.so"
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", str(lib), str(ROOT / "tests" / "hip_recorder.cpp")],
                   check=True)

    def run(code):
        p = subprocess.run([sys.executable, "-c", PRELUDE.format(recorder=str(lib), root=str(ROOT)) + code],
                           capture_output=True, text=True, timeout=300)
        assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-4000:]
        return p.stdout

    return run


@pytest.mark.parametrize("what", ["malloc", "copy"])
def test_a_failed_commit_leaves_no_copy_in_flight(recorded, what):
    """Small meshes are expanded into host arrays that the call owns: whichever allocation or
    copy of the commit fails, no copy may still read them when it returns."""
    out = recorded(f"""
failed, left = 0, []
for n in range(60):
    ctx = ohpt.Context(16, 16)
    ctx.begin_scene()
    rng = np.random.default_rng(0)
    for nt, world in ((7, None), (3000, 2 * np.eye(4)), (5, None), (2500, None), (4, None)):
        v = rng.random((nt + 2, 3), dtype=np.float32)
        ctx.add_mesh(v, rng.integers(0, nt + 2, (nt, 3)), normals=v, world=world)
    R.rec_fail_{what}(n)
    rc = ctx.L.ohpt_scene_commit(ctx.h)
    R.rec_fail_{what}(-1)
    if rc == 0:
        break
    failed += 1
    if R.rec_pending():
        left.append((n, R.rec_pending()))
    ctx.close()
print(rc, failed, left)
""")
    rc, failures, left = out.strip().split(" ", 2)
    assert int(rc) == 0 and int(failures) >= 10      # every one of them failed once, then none
    assert left == "[]", f"(failing one, copies in flight): {left}"


def test_a_failed_texture_upload_leaves_no_copy_in_flight(recorded):
    """The texels are the caller's, who may free them as soon as the call returns."""
    out = recorded("""
failed, left = 0, []
for update, n in [(u, k) for u in (False, True) for k in range(20)]:
    ctx = ohpt.Context(16, 16)
    t = np.ones((5, 7, 3) if n < 10 else (90, 100, 3), np.float32)   # packed on the host, on the device
    if update:
        ctx.upload_texture(t)
    R.rec_fail_copy(n % 10)
    try:
        ctx.update_texture(0, t) if update else ctx.upload_texture(t)
    except ohpt.OhptError:
        failed += 1
        if R.rec_pending():
            left.append((update, n, R.rec_pending()))
    R.rec_fail_copy(-1)
    ctx.close()
print(failed, left)
""")
    failures, left = out.strip().split(" ", 1)
    assert int(failures) >= 4
    assert left == "[]", f"(update, failing copy, copies in flight): {left}"


def test_ray_queries_keep_the_scratch_of_one_lane(recorded):
    """A context that only traces rays runs one traversal at a time; renders run three."""
    out = recorded("""
ctx = ohpt.Context(16, 16)
ctx.begin_scene()
ctx.add_mesh(np.eye(3, dtype=np.float32), [0, 1, 2])
ctx.commit_scene()
rays = np.ones((5, 8), np.float32)
held = [R.rec_allocated()]
for call in (ctx.trace_rays, ctx.occluded_rays, ctx.trace_rays):
    call(rays)
    held.append(R.rec_allocated() - held[0])
ctx.render(1)
ctx.trace_rays(rays)
held.append(R.rec_allocated() - held[0])
print(*held[1:])
""")
    one, two, three, rendered = map(int, out.split())
    # the recorder's device holds 256 x 2 blocks of 128 threads, with 72 stack slots of 4 bytes each
    lane = 256 * 2 * 128 * 72 * 4
    assert lane <= one < 1.2 * lane and one == two == three
    assert rendered >= 3 * lane


def test_a_render_that_ran_out_of_memory_can_be_followed_by_a_smaller_one(recorded):
    """Growing the path buffers frees the old ones first: after a failure half way, a render
    of the old size has to allocate again instead of using what is gone."""
    out = recorded("""
bad = []
for n in range(16):
    ctx = ohpt.Context(16, 16)
    ctx.begin_scene()
    ctx.add_mesh(np.eye(3, dtype=np.float32), [0, 1, 2])
    ctx.commit_scene()
    ctx.render(1)
    before = R.rec_allocated()
    assert ctx.L.ohpt_resize(ctx.h, 64, 64) == 0
    grown = R.rec_allocated() - before
    R.rec_fail_malloc(n)
    failed = ctx.L.ohpt_render(ctx.h, 1, 0) != 0
    R.rec_fail_malloc(-1)
    if not failed:
        break
    assert ctx.L.ohpt_resize(ctx.h, 16, 16) == 0
    ctx.render(1)
    if R.rec_allocated() < before + grown:
        bad.append(n)
    ctx.close()
print(n, bad)
""")
    n, bad = out.strip().split(" ", 1)
    assert int(n) >= 10 and bad == "[]", out


def test_staging_of_large_uploads_is_given_back(recorded):
    """Texels and vertices pass through a staging buffer: up to 256 MB of it stay with the
    context for the next upload, more is freed before the call returns."""
    out = recorded("""
def held(h, w, nv):
    # a texture upload, its update and a commit: what stays allocated beyond the texture and the scene
    ctx = ohpt.Context(16, 16)
    ctx.begin_scene()
    ctx.add_mesh(np.zeros((nv, 3), np.float32), np.arange(3 * 2048)[::-1] % nv)
    before = R.rec_allocated()
    ctx.commit_scene()
    scene = R.rec_allocated() - before
    t = np.zeros((h, w, 3), np.float32)
    before = R.rec_allocated()
    ctx.upload_texture(t)
    ctx.update_texture(0, t)
    texture = R.rec_allocated() - before - h * w * 16
    ctx.close()
    return scene, texture
print(*held(8, 8, 3 * 2048), *held(4800, 4800, 24 << 20))
""")
    scene, texture, large_scene, large_texture = map(int, out.split())
    assert abs(large_scene - scene) < (1 << 20), (scene, large_scene)
    assert abs(large_texture - texture) < (1 << 20), (texture, large_texture)


@pytest.mark.parametrize("h,w", [(1080, 1920), (1088, 1936), (736, 1024), (512, 768)])
def test_persistent_convolutions_fit_the_resident_blocks(recorded, h, w):
    """Two blocks per compute unit are resident: layers of at most twice as many tiles and channel
    groups run one block for each, larger ones as many blocks as are resident, which walk equal ranges."""
    out = recorded(f"""
d = ohpt.Denoiser(seed=1)
R.rec_clear_launches()
d.infer(np.zeros((1, {h}, {w}, 4), np.float32))
for name, g in launches():
    if "k_conv_ring" in name or "k_conv_dma" in name:
        print("ring" if "k_conv_ring" in name else "dma", *g)
""")
    got = [line.split() for line in out.strip().split("\n")]
    # level and groups of 32 output channels of the layers without an upsampled or feature input
    layers = [(1, 2), (1, 2), (2, 3), (2, 3), (3, 4), (3, 4), (4, 5), (4, 5), (3, 4), (2, 3), (1, 2)]
    up = lambda a, b: -(-a // b)
    assert len(got) == len(layers)
    for (level, groups), (kind, *grid) in zip(layers, got):
        x, y = up(up(w, 16) * 16 >> level, 16), up(up(h, 16) * 16 >> level, 16)
        if x * y * groups <= 2 * 512:
            assert (kind, list(map(int, grid))) == ("dma", [x, y, groups])
        else:
            ranges = up(x * y, up(x * y, 512 // groups))
            assert (kind, int(grid[0])) == ("ring", up(ranges * groups, 8) * 8)
            assert ranges * groups <= 512


def test_small_textures_launch_nothing(recorded):
    """Up to 8192 texels an update is one copy: the kernels' launches take longer than the loop."""
    out = recorded("""
for w in (1, 8192, 8193):
    ctx = ohpt.Context(16, 16)
    t = np.zeros((1, w, 3), np.float32)
    ctx.upload_texture(t)
    R.rec_clear_launches()
    ctx.update_texture(0, t)
    print(R.rec_launches())
""")
    assert out.split() == ["0", "0", "2"]


def test_small_gradients_launch_nothing(recorded):
    out = recorded("""
import dataclasses
for w in (1, 10240, 10241):
    sc = dataclasses.replace(S.lantern(freq=2, tex_size=64), textures=[np.zeros((1, w, 3), np.float32)], width=16, height=16)
    ctx = ohpt.Context(16, 16)
    ctx.load_scene(sc)
    ctx.adjoint(np.ones((16, 16, 4), np.float32), 1)
    R.rec_clear_launches()
    ctx.texture_gradient(0, (1, w, 3))
    print(R.rec_launches())
""")
    assert out.split() == ["0", "0", "1"]
