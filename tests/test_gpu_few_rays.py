"""The traversal with eight lanes per ray (few rays) against the oracle and against one lane per ray:
launches of one ray to more than one round of groups, deep stacks that leave LDS, never-cull slots,
both leaf tests."""
import numpy as np
import pytest

import oracle
import portablert_amd as prt
from conftest import load_golden
from helpers import assert_same
from test_gpu_build import rays_in, soup

pytestmark = pytest.mark.gpu

FULL = prt.mask_of(prt.ALL_TAGS)


def both(ctx, rays, want, what):
    """Eight lanes per ray (the automatic launch), then one (an explicit wave count)."""
    for waves in (0, 16):
        ctx.set_option("waves_per_cu", waves)
        try:
            assert_same(ctx.nearest_hits(rays, FULL), want, what=f"{what} waves={waves}")
        finally:
            ctx.set_option("waves_per_cu", 0)


@pytest.mark.parametrize("leaf_test", [0, 1])
@pytest.mark.parametrize("n", [1, 7, 9, 65, 4097, 65537, 98304])
def test_ray_counts(gpu_ctx, n, leaf_test):
    tris, rays = soup(3000, 1), rays_in(n, n)
    gpu_ctx.set_tris(tris)
    gpu_ctx.set_option("leaf_test", leaf_test)
    try:
        mode = oracle.LOWEST_ID | (oracle.WATERTIGHT if leaf_test else 0)
        both(gpu_ctx, rays, oracle.trace(tris, rays, mode), f"n={n} leaf_test={leaf_test}")
    finally:
        gpu_ctx.set_option("leaf_test", 0)


@pytest.mark.parametrize("name", ["sliver_gap", "sliver_cloud", "sliver_tilted", "stack", "soup200", "tie"])
@pytest.mark.parametrize("cull", [1, 0])
def test_fixtures(gpu_ctx, name, cull):
    g = load_golden("edge_" + name)
    gpu_ctx.set_tris(g["tris"])
    gpu_ctx.set_option("cull", cull)
    try:
        both(gpu_ctx, g["rays"], oracle.trace(g["tris"], g["rays"], oracle.LOWEST_ID), name)
    finally:
        gpu_ctx.set_option("cull", 1)


def test_stack_deeper_than_lds(gpu_ctx):
    """Equal triangles make a tree some 80 levels deep, and without culling every level's siblings
    wait on the stack: far more entries than LDS holds."""
    tris = np.concatenate([np.repeat(soup(1, 9) * 3, 600, axis=0), soup(200, 5)]).astype(np.float32)
    rays = rays_in(3000, 5)
    gpu_ctx.set_tris(tris)
    gpu_ctx.set_option("cull", 0)
    try:
        both(gpu_ctx, rays, oracle.brute(tris, rays), "deep")
    finally:
        gpu_ctx.set_option("cull", 1)


@pytest.mark.parametrize("leaf_test", [0, 1])
@pytest.mark.parametrize("n", [1, 4096, 4097, 65537, 98305, 131072, 131073])
def test_second_pass(gpu_ctx, n, leaf_test):
    """Rays with d_x = 0, which the second launch traces: listed, more than the list holds (4,096),
    more than one round of groups, and where its eight lanes per ray end; an ordinary ray in every 7."""
    tris, rays = soup(3000, 1), rays_in(n, n)
    rays[np.arange(n) % 7 != 3, 3] = 0.0
    gpu_ctx.set_tris(tris)
    gpu_ctx.set_option("leaf_test", leaf_test)
    try:
        mode = oracle.LOWEST_ID | (oracle.WATERTIGHT if leaf_test else 0)
        both(gpu_ctx, rays, oracle.trace(tris, rays, mode), f"n={n} leaf_test={leaf_test}")
    finally:
        gpu_ctx.set_option("leaf_test", 0)
