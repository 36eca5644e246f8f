"""Batch builds with few children a node, whose trees reach far below the level launches: records
equal the oracle's for every width and leaf size, scenes of 1 to 30,000 triangles."""
import numpy as np
import pytest
import torch

import oracle
import portablert_amd as prt
from helpers import assert_same
from test_gpu_build import rays_in, soup

pytestmark = pytest.mark.gpu

FULL = prt.mask_of(prt.ALL_TAGS)


@pytest.fixture(scope="module")
def scenes_and_hits():
    tris = [soup(n, n) for n in (30000, 1, 2, 3, 4097, 7, 600)]
    rays = [rays_in(500, len(t)) for t in tris]
    return tris, rays, np.concatenate([oracle.brute(t, r) for t, r in zip(tris, rays)])


@pytest.mark.parametrize("width", [2, 3, 4, 6, 8])
@pytest.mark.parametrize("leaf", [1, 2, 4])
def test_widths(gpu_ctx, scenes_and_hits, width, leaf):
    tris, rays, want = scenes_and_hits
    d_tris, d_rays = (torch.from_numpy(np.concatenate(x)).cuda() for x in (tris, rays))
    out = torch.zeros(len(d_rays) * prt.layout(FULL)[0], dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    batch = prt.Batch(gpu_ctx, list(map(len, tris)), list(map(len, rays)), FULL)
    was = [batch.params(k) for k in range(prt.BATCH_BUCKETS)]
    try:
        for k in range(prt.BATCH_BUCKETS):
            batch.set_params(k, (width, leaf, 64))
        for _ in range(2):
            out.zero_()
            torch.cuda.synchronize()
            batch.run(d_tris.data_ptr(), d_rays.data_ptr(), out.data_ptr())
            batch.check()
            assert_same(out.cpu().numpy().view(prt.hit_dtype(FULL)), want, what=f"width {width} leaf {leaf}")
    finally:
        for k in range(prt.BATCH_BUCKETS):
            batch.set_params(k, was[k])
