"""PRT_STAT_TRACE_MS of a host call is the traversal of rays and records in device memory, not their way
over the host link: it agrees with the device call's."""
import numpy as np
import pytest
import torch

import portablert_amd as prt
from portablert_amd import scenes

pytestmark = pytest.mark.gpu

FULL = prt.mask_of(prt.ALL_TAGS)


@pytest.mark.parametrize("n", [60000, 131072])
def test_host_and_device_calls_time_the_same(gpu_ctx, n):
    gpu_ctx.set_tris(scenes.scene(2))
    rays = scenes.rays(2, count=n)
    d = torch.from_numpy(rays).cuda()
    out = torch.empty(n * prt.layout(FULL)[0], dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    gpu_ctx.nearest_hits(rays[:10], FULL)  # a context's first host call goes another way
    host, device = [], []
    gpu_ctx.set_option("time_kernel", 1)
    try:
        for _ in range(20):
            got = gpu_ctx.nearest_hits(rays, FULL)
            host.append(gpu_ctx.stat("trace_ms"))
            gpu_ctx.nearest_hits_device(d.data_ptr(), n, FULL, out.data_ptr())
            device.append(gpu_ctx.stat("trace_ms"))
        gpu_ctx.synchronize()
    finally:
        gpu_ctx.set_option("time_kernel", 0)
    assert got.tobytes() == out.cpu().numpy().tobytes()
    print(f"{n} rays: host {min(host):.4f} ms, device {min(device):.4f} ms")
    assert min(host) < 1.3 * min(device)
