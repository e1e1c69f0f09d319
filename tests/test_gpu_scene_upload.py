"""Scene uploads that are expanded or summed on the device: meshes around the size
from which their vertices are gathered there, alone and mixed, against the same
triangles added as one flat mesh; environment tables around the 2048-value passes
against numpy's sequential sums."""
import numpy as np
import pytest

from ohao_engine_amd import ohpt
from ohao_engine_amd import scenes as S

pytestmark = pytest.mark.gpu

MOVE = np.array([[0.8, -0.6, 0, 0.3], [0.6, 0.8, 0, -0.2], [0, 0, 1.5, 0.1], [0, 0, 0, 1]], np.float32)


def mesh(n, seed, indexed, normals, uvs):
    """n triangles over shared vertices, or with their corners in order."""
    rng = np.random.default_rng(seed)
    nv = max(3, n // 2) if indexed else 3 * n
    f = (rng.integers(0, nv, 3 * n) if indexed else np.arange(3 * n)).astype(np.uint32)
    pos = rng.random((nv, 3), dtype=np.float32)
    return pos, f, rng.random((nv, 3), dtype=np.float32) if normals else None, \
        rng.random((nv, 2), dtype=np.float32) if uvs else None


def frame(build):
    sc = S.cornell_box(40, 40)
    ctx = ohpt.Context(40, 40)
    ctx.begin_scene()
    build(ctx)
    ctx.commit_scene()
    rng = np.random.default_rng(0)
    tex = rng.random((16, 16, 3), dtype=np.float32)
    mats = sc.materials[:2].copy()
    mats["emissive"] = 0
    mats["albedo_tex"] = 0
    mats["emissive"][1] = 3.0
    ctx.load_scene(S.Scene(**{**sc.__dict__, "textures": [tex], "materials": mats}), upload_geometry=False)
    ctx.render(2)
    out = ctx.read_accum()
    ctx.close()
    return out


CASES = [[(2047, True, True, True, None)], [(2048, True, True, True, MOVE)], [(2049, False, True, True, None)],
         [(2048, False, False, False, MOVE)],
         [(5, True, False, True, None), (3000, False, True, False, None), (2047, False, True, True, MOVE),
          (1, True, False, False, MOVE), (2048, True, False, True, None), (7, False, True, True, None)]]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_meshes_equal_their_flat_triangles(case):
    parts = [(mesh(n, 10 * case + k, ix, nr, uv), w) for k, (n, ix, nr, uv, w) in enumerate(CASES[case])]
    any_n, any_uv = (any(p[0][i] is not None for p in parts) for i in (2, 3))

    def meshes(ctx):
        for k, ((p, f, n, u), w) in enumerate(parts):
            ctx.add_mesh(p, f, normals=n, uvs=u, material_base=k % 2, world=w)

    def flat(ctx):
        P, N, U, M = [], [], [], []
        for k, ((p, f, n, u), w) in enumerate(parts):
            q = p[f].astype(np.float64)
            m = None if n is None else n[f].astype(np.float64)
            if w is not None:   # sums in the library's order
                a = np.asarray(w, np.float32).astype(np.float64)
                q = np.stack([a[r, 0] * q[:, 0] + a[r, 1] * q[:, 1] + a[r, 2] * q[:, 2] + a[r, 3] for r in range(3)], 1)
                if m is not None:
                    m = normal_matrix_times(a, m)
            q = q.astype(np.float32)
            if m is None:
                t = q.reshape(-1, 3, 3)
                e1, e2 = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
                g = np.stack([e1[:, 1] * e2[:, 2] - e1[:, 2] * e2[:, 1], e1[:, 2] * e2[:, 0] - e1[:, 0] * e2[:, 2],
                              e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0]], 1)
                m = np.repeat(g, 3, 0)
            P.append(q)
            N.append(m.astype(np.float32))
            U.append(np.zeros((len(f), 2), np.float32) if u is None else u[f])
            M.append(np.full(len(f) // 3, k % 2, np.uint32))
        P, N, U = np.concatenate(P), np.concatenate(N), np.concatenate(U)
        ctx.add_mesh(P, np.arange(len(P), dtype=np.uint32), normals=N if any_n else None, uvs=U if any_uv else None,
                     mat_ids=np.concatenate(M))

    assert np.array_equal(frame(meshes), frame(flat))


def normal_matrix_times(a, v):
    """The inverse transpose by cofactors, each sum in the library's order."""
    (A, B, C), (D, E, F), (G, H, I) = a[0, :3], a[1, :3], a[2, :3]
    det = A * (E * I - F * H) - B * (D * I - F * G) + C * (D * H - E * G)
    n = np.array([[(E * I - F * H) / det, -(D * I - F * G) / det, (D * H - E * G) / det],
                  [-(B * I - C * H) / det, (A * I - C * G) / det, -(A * H - B * G) / det],
                  [(B * F - C * E) / det, -(A * F - C * D) / det, (A * E - B * D) / det]])
    return np.stack([n[r, 0] * v[:, 0] + n[r, 1] * v[:, 1] + n[r, 2] * v[:, 2] for r in range(3)], 1)


@pytest.mark.parametrize("W,H", [(1, 1), (5, 3), (255, 257), (2048, 2), (2051, 7), (4100, 5), (3, 2050)])
def test_environment_tables(W, H):
    rng = np.random.default_rng(W + H)
    env = rng.random((H, W, 4), dtype=np.float32)
    if H > 2:
        env[1] = 0.0                              # a black row
    ctx = ohpt.Context(16, 16)
    ctx.set_env(env)
    marg, cond, integral = ctx.export_env_cdf(W, H)[:3]
    ctx.close()
    f = np.float32
    theta = (f(np.pi) * (np.arange(H, dtype=f) + f(0.5))) / f(H)
    lum = (f(0.2126) * env[..., 0] + f(0.7152) * env[..., 1]) + f(0.0722) * env[..., 2]
    rows = np.cumsum(lum * np.sin(theta)[:, None].astype(f), axis=1, dtype=f)
    total = np.cumsum(rows[:, -1], dtype=f)
    want = np.where(rows[:, -1:] > 0, rows / np.maximum(rows[:, -1:], f(1e-30)), np.arange(1, W + 1, dtype=f) / f(W))
    # the sums run in one order; only the sine differs, by an ulp or two, and mostly cancels
    np.testing.assert_allclose(cond.reshape(H, W), want, rtol=1e-6)
    np.testing.assert_allclose(marg, total / total[-1], rtol=1e-6)
    np.testing.assert_allclose(integral, total[-1], rtol=1e-6)
