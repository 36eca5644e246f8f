"""The host-buffer call where its way to and from the GPU changes: rays read and records written in
pinned memory by the kernel, staged slices, chunks, and buffers that are pinned already."""
import numpy as np
import pytest
import torch

import portablert_amd as prt
from portablert_amd import scenes

pytestmark = pytest.mark.gpu

ALL = prt.mask_of(prt.ALL_TAGS)


@pytest.fixture(scope="module")
def room(gpu_ctx):
    gpu_ctx.set_tris(scenes.scene(2))
    return scenes.rays(2, first=1000, count=1100000)


def device_records(ctx, rays, mask):
    d = torch.from_numpy(rays).cuda()
    out = torch.empty(len(rays) * prt.layout(mask)[0], dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    ctx.nearest_hits_device(d.data_ptr(), len(rays), mask, out.data_ptr())
    torch.cuda.synchronize()
    return out.cpu().numpy().tobytes()


@pytest.mark.parametrize("mask", [ALL, prt.VALID])
@pytest.mark.parametrize("n", [1, 131071, 131072, 131073, 200001, 1048576, 1048577])
def test_host_call_equals_device_call(gpu_ctx, room, n, mask):
    rays = np.ascontiguousarray(room[:n])
    assert gpu_ctx.nearest_hits(rays, mask).tobytes() == device_records(gpu_ctx, rays, mask)


def test_pinned_rays_and_changing_sizes(gpu_ctx, room):
    """Rays in memory that HIP knows, and small calls after large ones (kept buffers)."""
    for n in (200001, 777, 131072, 3):
        rays = torch.from_numpy(np.ascontiguousarray(room[:n])).pin_memory().numpy()
        assert gpu_ctx.nearest_hits(rays, ALL).tobytes() == device_records(gpu_ctx, rays, ALL)
