"""Rays with zero direction components through vertices, edges and insides of a mesh, with the
default distance culling: equal to the oracle, also where a wall that runs along the ray has a
determinant of rounding errors and a t far from its box."""
import numpy as np
import pytest

import oracle
import portablert_amd as prt
from helpers import assert_same
from portablert_amd import scenes

pytestmark = pytest.mark.gpu

FULL = prt.mask_of(prt.ALL_TAGS)


def turned(tris, axis, angle):
    """Turned about an axis in 64 bits: walls along it stay so but for the last bits."""
    i, j = [k for k in range(3) if k != axis]
    v = tris.reshape(-1, 3).astype(np.float64)
    x, y = v[:, i].copy(), v[:, j].copy()
    v[:, i], v[:, j] = np.cos(angle) * x - np.sin(angle) * y, np.sin(angle) * x + np.cos(angle) * y
    return v.astype(np.float32).reshape(-1, 9)


def aimed(rng, tris, n):
    """Rays with every pattern of one or two zero components, whose line passes exactly (in those
    coordinates) through a vertex, a point of an edge or of the inside of some triangle."""
    ext = float(np.ptp(tris.reshape(-1, 3), axis=0).max())
    d = rng.normal(size=(n, 3))
    pattern = rng.integers(1, 7, n)
    for k in range(3):
        d[(pattern >> k & 1) == 1, k] = 0
    w = rng.dirichlet((1, 1, 1), n)
    kind = rng.integers(0, 3, n)
    w[kind == 0] = (1, 0, 0)
    w[kind == 1, 2] = 0
    w[kind == 1, 1] = 1 - w[kind == 1, 0]
    p = (tris[rng.integers(0, len(tris), n)].reshape(n, 3, 3) * w[:, :, None]).sum(1)
    o = p - d * rng.uniform(.003, .6, (n, 1)) * ext
    o = np.where(d == 0, p, o)
    return np.concatenate([o, d], 1).astype(np.float32)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("scene", ["room", "blocks"])
def test_aimed_axis_rays(gpu_ctx, scene, axis):
    rng = np.random.default_rng(axis + 10 * len(scene))
    if scene == "room":
        tris = scenes.scene(2)
    else:
        tris = ((rng.integers(-40, 41, (20000, 1, 3)) + rng.integers(-6, 7, (20000, 3, 3))) / 16).reshape(-1, 9)
    tris = turned(tris.astype(np.float32), axis, .3 + axis)
    rays = aimed(rng, tris, 150000)
    gpu_ctx.set_tris(tris)
    got = gpu_ctx.nearest_hits(rays, FULL)
    few = gpu_ctx.nearest_hits(rays[:60000], FULL)  # eight lanes a ray
    assert few.tobytes() == got[:60000].tobytes()
    gpu_ctx.set_option("cull", 0)
    try:
        assert_same(got, gpu_ctx.nearest_hits(rays, FULL), what="against the exact mode")
    finally:
        gpu_ctx.set_option("cull", 1)
    some = rng.choice(len(rays), 2000, replace=False)
    assert_same(got[some], oracle.brute(tris, rays[some]), what="against the oracle")
