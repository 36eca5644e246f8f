"""The clustered build with more workgroups than the chip holds at once, where the clustering ends:
its last launches start workgroups while the first one reports that few clusters are left."""
import time

import numpy as np
import pytest

import oracle
import portablert_amd as prt
from helpers import assert_same
from test_gpu_build import rays_in, soup

pytestmark = pytest.mark.gpu


def test_equal_triangles_are_refused_early(gpu_ctx):
    """They merge one pair a step into a chain that no tree of 128 levels holds: refused after 4,096
    steps (some 0.1 s), not after one for every triangle (seconds)."""
    tris = np.repeat(soup(1, 9), 400000, axis=0)
    t0 = time.monotonic()
    with pytest.raises(prt.PrtError) as e:
        gpu_ctx.set_tris(tris)
    assert time.monotonic() - t0 < 1.5
    assert e.value.code == prt.ERR_HIP
    gpu_ctx.set_tris(soup(100, 9))  # the context still builds


@pytest.mark.parametrize("n", [600001, 1000003, 1900001])
def test_builds_agree(gpu_ctx, n):
    tris, rays = soup(n, n), rays_in(64, n)
    want = oracle.brute(tris, rays)
    for k in range(3):
        gpu_ctx.set_tris(tris)
        assert_same(gpu_ctx.nearest_hits(rays, prt.mask_of(prt.ALL_TAGS)), want, what=f"n={n} build {k}")
