"""Rays with zero direction components: quantized and fp32 nodes, with and without distance culling,
both leaf tests, after a build and after a refit, equal to the oracle's brute force bit for bit.
Half of the origins and every vertex lie on a coarse grid, so origins on box sides (where the
reference slab test meets 0 * inf) and on the low x side of a triangle are common."""
import numpy as np
import pytest

import oracle
import portablert_amd as prt
from helpers import assert_same

pytestmark = pytest.mark.gpu

FULL = prt.mask_of(prt.ALL_TAGS)


def grid_soup(rng, n, size):
    c = rng.integers(-24, 25, (n, 1, 3))
    return ((c + rng.integers(-size, size + 1, (n, 3, 3))) / 16.0).reshape(n, 9).astype(np.float32)


def axis_rays(rng, n):
    """Every pattern of zero components (of either sign), no direction at all among them, and NaN."""
    r = rng.uniform(-2, 2, (n, 6)).astype(np.float32)
    on = rng.random(n) < 0.5
    r[on, :3] = (rng.integers(-32, 33, (on.sum(), 3)) / 16.0).astype(np.float32)
    pattern = rng.integers(1, 8, n)
    for k in range(3):
        z = (pattern >> k & 1) == 1
        r[z, 3 + k] = np.where(rng.random(z.sum()) < 0.5, np.float32(0.0), np.float32(-0.0))
    r[::97, rng.integers(0, 6)] = np.nan
    r[5::101, 3] = np.float32(1e-30)  # neither zero nor in the range of the one-fma test
    return r


def one_nan(hits):
    """A NaN's sign and payload depend on the processor: every NaN as the same one."""
    hits = hits.copy()
    for f in ("t", "u", "v", "px", "py", "pz"):
        hits[f][np.isnan(hits[f])] = np.nan
    return hits


@pytest.mark.parametrize("leaf_test", [0, 1])
@pytest.mark.parametrize("n,size", [(1, 8), (37, 12), (2000, 3)])
def test_axis_rays_equal_brute_force(gpu_ctx, n, size, leaf_test):
    rng = np.random.default_rng(n + leaf_test)
    tris, rays = grid_soup(rng, n, size), axis_rays(rng, 20000)
    moved = grid_soup(rng, n, size)
    mode = oracle.LOWEST_ID | (oracle.WATERTIGHT if leaf_test else 0)
    try:
        gpu_ctx.set_option("leaf_test", leaf_test)
        for what, scene in (("build", tris), ("refit", moved)):
            want = one_nan(oracle.brute(scene, rays, mode=mode))
            gpu_ctx.set_tris(scene) if what == "build" else gpu_ctx.refit(scene)
            for fmt in (1, 0):
                for cull in (1, 0):
                    gpu_ctx.set_option("node_format", fmt)
                    gpu_ctx.set_option("cull", cull)
                    assert_same(one_nan(gpu_ctx.nearest_hits(rays, FULL)), want,
                                what=f"{what} n={n} leaf_test={leaf_test} fmt={fmt} cull={cull}")
    finally:
        for name, v in (("leaf_test", 0), ("node_format", 1), ("cull", 1)):
            gpu_ctx.set_option(name, v)


def test_orthographic_view_far_coordinates(gpu_ctx):
    """A pixel grid along each axis over a soup far from the coordinate origin."""
    rng = np.random.default_rng(3)
    tris = (rng.uniform(-1, 1, (3000, 1, 3)) + rng.uniform(-.05, .05, (3000, 3, 3)) + 1000.0).reshape(-1, 9)
    tris = tris.astype(np.float32)
    gpu_ctx.set_tris(tris)
    for axis in range(3):
        for sign in (1.0, -1.0):
            rays = np.zeros((4096, 6), np.float32)
            rays[:, :3] = rng.uniform(999, 1001, (4096, 3))
            rays[:, axis] = 1000.0 - 3.0 * sign
            rays[:, 3 + axis] = sign
            rays[::3, axis] = 1000.0
            assert_same(gpu_ctx.nearest_hits(rays, FULL), oracle.brute(tris, rays), what=f"axis {axis} {sign}")


@pytest.mark.parametrize("n_rays", [900, 6000])
def test_axis_rays_in_a_batch(gpu_ctx, n_rays):
    """Rays of three scenes that the first pass leaves to the second: few enough to be listed, and
    more than the list holds."""
    import torch
    rng = np.random.default_rng(n_rays)
    tris = [grid_soup(rng, n, 4) for n in (300, 1, 700)]
    rays = [axis_rays(rng, n) for n in (n_rays, 50, n_rays)]
    d_tris, d_rays = (torch.from_numpy(np.concatenate(x)).cuda() for x in (tris, rays))
    size, _ = prt.layout(FULL)
    out = torch.zeros(sum(map(len, rays)) * size, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    batch = prt.Batch(gpu_ctx, list(map(len, tris)), list(map(len, rays)), FULL)
    batch.capture(d_tris.data_ptr(), d_rays.data_ptr(), out.data_ptr())
    want = one_nan(np.concatenate([oracle.brute(t, r) for t, r in zip(tris, rays)]))
    for _ in range(3):  # every replay takes the second pass again
        out.zero_()
        torch.cuda.synchronize()
        batch.replay()
        batch.check()
        assert_same(one_nan(out.cpu().numpy().view(prt.hit_dtype(FULL))), want, what=f"batch {n_rays}")
