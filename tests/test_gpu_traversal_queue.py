"""The traversal's leaf queue, stack and ray dealing against the sequential oracle,
bit for bit: triangles that all overlap (four leaf hits in one node, a stack deeper
than its LDS part), origins on box planes, distances from below zero, and ray
counts around the blocks, the resident threads and the 64 fetch groups. Batches that
are resident at once take the kernel with a ray per thread, larger ones the
persistent one with the queue: each scene goes through both."""
import re
from pathlib import Path

import numpy as np
import pytest

from ohao_engine_amd import ohpt
from ohao_engine_amd import scenes as S

pytestmark = pytest.mark.gpu


def scene(pos):
    return S.Scene(pos=np.ascontiguousarray(pos, np.float32), mat=np.zeros(len(pos), np.uint32),
                   materials=S.cornell_box().materials[:1], camera=S.cornell_box().camera)


def overlapping(n, seed):
    """Triangles that each span most of the unit cube."""
    return np.random.default_rng(seed).random((n, 9), dtype=np.float32)


def rays_in(lo, hi, n, seed, tmin=0.0, tmax=np.inf):
    rng = np.random.default_rng(seed)
    r = np.empty((n, 8), np.float32)
    r[:, 0:3] = rng.uniform(lo, hi, (n, 3))
    d = rng.standard_normal((n, 3))
    axis = rng.random(n) < 0.2                  # along an axis: slabs of zero extent in two of them
    d[axis] = np.eye(3)[rng.integers(0, 3, axis.sum())] * rng.choice([-1.0, 1.0], (axis.sum(), 1))
    r[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 3] = tmin
    r[:, 7] = tmax
    return r


RESIDENT = 327680   # threads of a 256-CU grid


def check(oracle, pos, rays):
    sc = scene(pos)
    o = oracle.OracleScene(sc)
    want, visits, _ = o.trace(rays)
    occluded = o.occluded(rays)
    ctx = ohpt.Context(32, 32)
    ctx.load_scene(sc)
    # once as they are, and over and over in another order until they are more than are resident
    order = np.concatenate([np.random.default_rng(k).permutation(len(rays)) for k in range(RESIDENT // len(rays) + 1)])
    for batch in (np.arange(len(rays)), order[:RESIDENT + 1001] if len(rays) > 1 else order[:0]):
        if len(batch):
            assert np.array_equal(ctx.trace_rays(rays[batch]).view(np.uint32), want[batch].view(np.uint32))
            assert np.array_equal(ctx.occluded_rays(rays[batch]), occluded[batch])
    ctx.close()
    return visits


@pytest.mark.parametrize("n", [1, 2, 3, 5, 17, 300, 20000])
def test_overlapping_triangles(oracle, n):
    print(f"overlapping {n}", flush=True)
    pos = overlapping(n, n)
    visits = check(oracle, pos, rays_in(-0.5, 1.5, 3000, n))
    if n == 20000:
        assert visits.max() > 200


@pytest.mark.parametrize("tmin,tmax", [(-2.0, 3.0), (0.25, 0.75), (0.0, 0.0), (-1.0, -0.1)])
def test_distance_ranges(oracle, tmin, tmax):
    print(f"range {tmin} {tmax}", flush=True)
    check(oracle, overlapping(500, 9), rays_in(0.0, 1.0, 4000, 5, tmin, tmax))


def test_origins_on_box_planes(oracle):
    pos = np.round(overlapping(400, 3) * 8) / 8        # boxes on a grid, and the origins too
    rays = rays_in(0.0, 1.0, 6000, 7)
    rays[:, 0:3] = np.round(rays[:, 0:3] * 8) / 8
    check(oracle, pos, rays)


@pytest.mark.parametrize("n", [1, 63, 64, 129, 327679, 327680, 327681, 327680 + 64 * 64 + 1, 700001])
def test_ray_counts(oracle, n):
    """A 256-CU grid holds 327,680 threads; further rays are dealt in 64 groups."""
    print(f"count {n}", flush=True)
    sc = S.displaced_sphere(6, 0.2, 1)
    V, F = sc[0], sc[3]
    check(oracle, V[F.reshape(-1)].reshape(-1, 9), rays_in(-1.2, 1.2, n, n))


def stack_depth(nodes, ray, t_hit):
    """Entries on the stack where `ray` needs most, with every box behind its hit culled from
    the start: any traversal in this order holds these, and more while its hit is farther."""
    box = nodes[:, :24].view(np.float32).astype(np.float64).reshape(-1, 2, 3, 4)
    origin, d = ray[0:3].astype(np.float64), ray[4:7].astype(np.float64)
    inv = 1.0 / np.where(np.abs(d) < 1e-20, 1e-20, d)
    stack, deepest = [0], 0
    while stack:
        n = stack.pop()
        t = (box[n] - origin[:, None]) * inv[:, None]
        near = np.maximum(np.minimum(t[0], t[1]).max(0), ray[3])
        far = np.minimum(np.maximum(t[0], t[1]).min(0), t_hit * (1 - 1e-6))
        stack += [int(nodes[n, 24 + k]) for k in np.argsort(-near)
                  if near[k] <= far[k] and nodes[n, 24 + k] < 0x80000000]
        deepest = max(deepest, len(stack))
    return deepest


def test_stack_deeper_than_its_lds_part(oracle):
    """The rays with most visits of the 20,000 overlapping triangles spill to global memory."""
    header = Path(ohpt.__file__).parent / "csrc" / "ohpt_internal.h"
    lds = int(re.search(r"#define OHPT_STACK_LDS (\d+)", header.read_text()).group(1))
    pos, rays = overlapping(20000, 20000), rays_in(-0.5, 1.5, 3000, 20000)
    visits = check(oracle, pos, rays)
    rays = rays[np.argsort(-visits.astype(np.int64))[:20]]
    ctx = ohpt.Context(32, 32)
    ctx.load_scene(scene(pos))
    hits, nodes = ctx.trace_rays(rays), ctx.export_bvh4()
    ctx.close()
    t = np.where(hits[:, 1].view(np.uint32) == 0xFFFFFFFF, np.inf, hits[:, 0])
    depths = [stack_depth(nodes, r, v) for r, v in zip(rays, t)]
    print(f"stack depths {sorted(depths)} with {lds} entries in LDS", flush=True)
    assert sum(d - 1 > lds for d in depths) >= 10   # the nearest child may be kept in a register
