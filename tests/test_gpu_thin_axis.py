"""Rays with zero direction components against triangles that are thin, near coordinate 0, on the zero
axes: records equal the oracle's brute force in every mode that takes the one-fma node test."""
import numpy as np
import pytest

import oracle
import portablert_amd as prt
from helpers import assert_same
from test_one_fma_rays import THIN, huge_directions, squeezed, swap_yz

pytestmark = pytest.mark.gpu

FULL = prt.mask_of(prt.ALL_TAGS)
DEFAULTS = (("leaf_test", 0), ("node_format", 1), ("cull", 1), ("waves_per_cu", 0))


def thin_pairs():
    """(triangle, rays): y and z exchanged, both signs of the zero components."""
    for t, r in THIN:
        for swapped in (False, True):
            rays = np.stack([np.asarray(r, np.float32)] * 2)
            if swapped:
                rays = np.stack([swap_yz(x) for x in rays])
            for k, zero in enumerate((0.0, -0.0)):
                rays[k, 3:][rays[k, 3:] == 0] = zero
            yield (swap_yz(t) if swapped else np.asarray(t, np.float32)).reshape(1, 9), rays


def options(ctx, **kw):
    for name, v in {**dict(DEFAULTS), **kw}.items():
        ctx.set_option(name, v)


@pytest.mark.parametrize("leaf_test", [0, 1])
@pytest.mark.parametrize("waves", [0, 16])
def test_thin_triangles(gpu_ctx, waves, leaf_test):
    mode = oracle.LOWEST_ID | (oracle.WATERTIGHT if leaf_test else 0)
    try:
        for i, (tri, rays) in enumerate(thin_pairs()):
            want = oracle.brute(tri, rays, mode=mode)
            gpu_ctx.set_tris(tri)
            for fmt in (1, 0):
                for cull in (1, 0):
                    options(gpu_ctx, leaf_test=leaf_test, node_format=fmt, cull=cull, waves_per_cu=waves)
                    assert_same(gpu_ctx.nearest_hits(rays, FULL), want, what=f"pair {i} fmt={fmt} cull={cull}")
    finally:
        options(gpu_ctx)


@pytest.mark.parametrize("n_rays", [4000, 98305])
def test_squeezed_scene(gpu_ctx, n_rays):
    """Many such triangles together, by eight lanes a ray and by one, without distance culling."""
    tris, rays = squeezed(np.random.default_rng(7), 300)
    rays = np.resize(rays, (n_rays, 6))
    want = oracle.brute(tris, rays)
    gpu_ctx.set_tris(tris)
    try:
        for waves in (0, 16):
            options(gpu_ctx, cull=0, waves_per_cu=waves)
            assert_same(gpu_ctx.nearest_hits(rays, FULL), want, what=f"waves={waves}")
    finally:
        options(gpu_ctx)


def test_huge_directions_without_culling(gpu_ctx):
    """t down to the denormals, where the one-fma test's margins end: the reference formula's rays."""
    tris, rays = huge_directions(np.random.default_rng(11), 400)
    rays = np.resize(rays, (8000, 6))
    want = oracle.brute(tris, rays)
    gpu_ctx.set_tris(tris)
    try:
        for waves in (0, 16):
            options(gpu_ctx, cull=0, waves_per_cu=waves)
            assert_same(gpu_ctx.nearest_hits(rays, FULL), want, what=f"waves={waves}")
    finally:
        options(gpu_ctx)


def test_thin_triangles_in_a_batch(gpu_ctx):
    import torch
    pairs = list(thin_pairs())
    d_tris, d_rays = (torch.from_numpy(np.concatenate(x)).cuda() for x in zip(*pairs))
    out = torch.zeros(len(d_rays) * prt.layout(FULL)[0], dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    batch = prt.Batch(gpu_ctx, [1] * len(pairs), [2] * len(pairs), FULL)
    batch.run(d_tris.data_ptr(), d_rays.data_ptr(), out.data_ptr())
    batch.check()
    want = np.concatenate([oracle.brute(t, r) for t, r in pairs])
    assert_same(out.cpu().numpy().view(prt.hit_dtype(FULL)), want, what="batch")
