"""The clustered build at the sizes where its kernels change: one workgroup (up to 1,024
triangles), small tiles (up to 40,000 clusters), whole tiles, the tile counts scanned by launches of
their own (above 4,096 tiles), and inputs that merge slower than the build guesses."""
import numpy as np
import pytest

import oracle
import portablert_amd as prt
from helpers import assert_same
from test_gpu_parity import check_bvh

pytestmark = pytest.mark.gpu

FULL = prt.mask_of(prt.ALL_TAGS)


def soup(n, seed):
    rng = np.random.default_rng(seed)
    size = 0.5 * max(1.0, n) ** (-1 / 3)
    return (rng.uniform(-1, 1, (n, 1, 3)) + rng.uniform(-size, size, (n, 3, 3))).reshape(n, 9).astype(np.float32)


def rays_in(n, seed):
    rng = np.random.default_rng(seed + 1)
    d = rng.normal(size=(n, 3))
    return np.concatenate([rng.uniform(-1, 1, (n, 3)), d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)


@pytest.mark.parametrize("collapse", [1, 0])
@pytest.mark.parametrize("n", [1, 2, 3, 33, 1023, 1024, 1025, 4999, 39999, 40001, 100003])
def test_sizes(gpu_ctx, n, collapse):
    tris, rays = soup(n, n), rays_in(2000, n)
    try:
        gpu_ctx.set_option("collapse", collapse)
        gpu_ctx.set_tris(tris)
        check_bvh(gpu_ctx, tris)
        assert_same(gpu_ctx.nearest_hits(rays, FULL), oracle.brute(tris, rays), what=f"n={n} collapse={collapse}")
        gpu_ctx.refit(soup(n, n + 7))  # the level starts come from the build
        assert_same(gpu_ctx.nearest_hits(rays, FULL), oracle.brute(soup(n, n + 7), rays), what=f"refit n={n}")
    finally:
        gpu_ctx.set_option("collapse", 1)


def test_more_tiles_than_a_step_sums(gpu_ctx):
    n = 4096 * 480 + 1
    tris, rays = soup(n, 5), rays_in(64, 5)
    gpu_ctx.set_tris(tris)
    assert_same(gpu_ctx.nearest_hits(rays, FULL), oracle.brute(tris, rays), what="large")


def test_slow_merging(gpu_ctx):
    """Groups of equal triangles merge one pair a step: more steps than the guess, and more levels."""
    groups = np.repeat(soup(8, 3) * 4, 500, axis=0).astype(np.float32)
    tris, rays = np.concatenate([groups, soup(300, 4)]), rays_in(500, 3)
    gpu_ctx.set_tris(tris)
    check_bvh(gpu_ctx, tris)
    assert_same(gpu_ctx.nearest_hits(rays, FULL), oracle.brute(tris, rays), what="equal triangles")
    gpu_ctx.refit(tris * np.float32(1.5))  # a level is one to a few nodes here, 80 levels deep
    check_bvh(gpu_ctx, tris * np.float32(1.5))
    assert_same(gpu_ctx.nearest_hits(rays, FULL), oracle.brute(tris * np.float32(1.5), rays), what="refit of a deep tree")
