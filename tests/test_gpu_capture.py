"""Traversals recorded into a graph: the first one of a context, uncaptured calls before its first
replay, and uncaptured calls between replays."""
import numpy as np
import pytest

import oracle
import portablert_amd as prt
from helpers import assert_same
from test_gpu_build import rays_in, soup

pytestmark = pytest.mark.gpu

FULL = prt.mask_of(prt.ALL_TAGS)


class Call:
    """Device rays with d_x = 0 among them (both launches of a traversal trace some), and records."""

    def __init__(self, tris, n, seed):
        import torch
        rays = rays_in(n, seed)
        rays[::5, 3] = 0
        self.want, self.n = oracle.brute(tris, rays), n
        self.rays = torch.from_numpy(rays).cuda()
        self.out = torch.zeros(n * prt.layout(FULL)[0], dtype=torch.uint8, device="cuda")

    def run(self, ctx, stream):
        ctx.nearest_hits_device(self.rays.data_ptr(), self.n, FULL, self.out.data_ptr(), stream.cuda_stream)

    def check(self, ctx, what):
        import torch
        torch.cuda.synchronize()
        ctx.synchronize()
        assert_same(self.out.cpu().numpy().view(prt.hit_dtype(FULL)), self.want, what=what)
        self.out.zero_()
        torch.cuda.synchronize()


def test_captured_learned_call_outlives_a_change_of_seeds(gpu_ctx):
    """A graph with a one-seed learned call replays after an uncaptured call of as many rays with four
    seeds: the predictions' buffer has not moved."""
    import torch
    tris = soup(3000, 31)
    gpu_ctx.set_tris(tris)
    prt.learned_setup(gpu_ctx, seed=1)
    call, stream, graph = Call(tris, 20000, 32), torch.cuda.Stream(), torch.cuda.CUDAGraph()

    def learned():
        prt.nearest_hits_learned_device(gpu_ctx, call.rays.data_ptr(), call.n, FULL, call.out.data_ptr(),
                                        stream.cuda_stream)
    try:
        learned()
        call.check(gpu_ctx, "one seed")
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
            learned()
        for k in range(3):
            gpu_ctx.set_option("seeds", 4)
            learned()
            call.check(gpu_ctx, f"four seeds, before replay {k}")
            gpu_ctx.set_option("seeds", 1)
            with torch.cuda.stream(stream):
                graph.replay()
            call.check(gpu_ctx, f"replay {k}")
    finally:
        gpu_ctx.set_option("seeds", 1)


@pytest.mark.parametrize("n", [1000, 120000])
def test_first_traversal_is_captured(n):
    import torch
    # no fresh device memory that happens to be 0: what an allocation of the counters may return
    junk = [torch.full((1 << 16,), 0x7F, dtype=torch.uint8, device="cuda") for _ in range(64)]
    torch.cuda.synchronize()
    del junk
    torch.cuda.empty_cache()
    tris = soup(500, 21)
    ctx = prt.Context(0)
    ctx.set_tris(tris)
    in_graph, eager = Call(tris, n, 22), Call(tris, n // 2 + 3, 23)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        in_graph.run(ctx, stream)
    ctx.synchronize()  # no error flags of a launch that has not run
    for k in range(2):
        eager.run(ctx, stream)
        eager.check(ctx, f"uncaptured call {k} before the first replay")
    for k in range(3):
        with torch.cuda.stream(stream):
            graph.replay()
        in_graph.check(ctx, f"replay {k}")
        eager.run(ctx, stream)
        eager.check(ctx, f"uncaptured call after replay {k}")
    ctx.close()
