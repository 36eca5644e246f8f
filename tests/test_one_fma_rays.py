"""Which rays take the one-fma node test (common.h, built here for the host), against the reference's
own slab and leaf test: a ray that takes it must enter the quantized box of every triangle that it
hits. The box test is restated in numpy with the kernels' roundings. No GPU."""
import ctypes
import subprocess

import numpy as np
import pytest

import oracle
import portablert_amd.build as build

F = np.float32

SRC = """
#include "common.h"
extern "C" void one_fma(const float *rays, const float *reach, int n, int exact, unsigned char *fast) {
	for (int i = 0; i < n; ++i) {
		const float *o = rays + 6 * i, *d = o + 3;
		const float inv[3] = {1.0f / d[0], 1.0f / d[1], 1.0f / d[2]};
		fast[i] = prt::ray_in_range(o, d, inv, reach[i]) && prt::one_fma_ray(o, d, inv, reach[i], exact);
	}
}
"""


@pytest.fixture(scope="module")
def one_fma(tmp_path_factory):
    d = tmp_path_factory.mktemp("one_fma")
    src, so = d / "one_fma.hip", d / "one_fma.so"
    src.write_text(SRC)
    subprocess.run([build.HIPCC, "--offload-host-only", "-std=c++17", "-O2", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I" + build.CSRC, str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))

    def f(rays, reach, exact=True):
        rays, reach = np.ascontiguousarray(rays, F), np.ascontiguousarray(reach, F)
        out = np.zeros(len(rays), np.uint8)
        lib.one_fma(*(a.ctypes.data_as(ctypes.c_void_p) for a in (rays, reach)), len(rays), exact,
                    out.ctypes.data_as(ctypes.c_void_p))
        return out.astype(bool)
    return f


def fma(a, b, c):
    return (np.asarray(a, np.float64) * b + c).astype(F)


def grid(lo, hi):
    """p + q 2^e grid of a box (grid_exp in build.hip): 2^e."""
    ext = hi - lo
    e = np.where(ext > 0, np.frexp(ext / F(255))[1] - 1, -126).clip(-126, 127)
    for _ in range(4):
        e = np.where((e < 127) & (fma(255, np.ldexp(F(1), e), lo) < hi), e + 1, e)
    return np.ldexp(F(1), e).astype(F)


def enters(tris, rays):
    """The one-fma test of the only child (the triangle's box) of a one-triangle scene's root."""
    v = tris.reshape(-1, 3, 3)
    lo, hi = v.min(1), v.max(1)
    s = grid(lo, hi)
    q = np.ceil((hi - lo) / s).clip(0, 255).astype(F)
    for _ in range(4):
        q = np.where((q < 255) & (fma(q, s, lo) < hi), q + 1, q)
    o, d = rays[:, :3], rays[:, 3:]
    with np.errstate(all="ignore"):
        inv = np.where(d == 0, np.copysign(F(2.0 ** 60), d), F(1) / d).astype(F)
        step, base = s * inv, (lo - o) * inv
        margin = (F(2.0 ** -18) * np.abs(inv)) * fma(255, s, np.abs(lo) + np.abs(o))
        qn, qf = np.where(inv >= 0, F(0), q), np.where(inv >= 0, q, F(0))
        near, far = fma(qn, step, base - margin).max(1), fma(qf, step, base + margin).min(1)
    return (far >= 0) & (near <= far)


def reference_hits(tris, rays):
    return np.array([oracle.brute(t, r)["t"][0] < np.inf for t, r in zip(tris, rays)])


def check(one_fma, tris, rays, exact=False):
    tris, rays = np.asarray(tris, F), np.asarray(rays, F)
    fast = one_fma(rays, np.abs(tris).max(1), exact)
    hit = reference_hits(tris, rays)
    assert hit.mean() > 0.2  # the inputs reach their triangles
    lost = fast & hit & ~enters(tris, rays)
    i = int(np.flatnonzero(lost)[0]) if lost.any() else 0
    assert not lost.any(), f"{lost.sum()} hits lost, first: triangle {tris[i]} ray {rays[i]}"


# Triangles thin and near coordinate 0 on a zero axis of the ray, which the box test left out when the
# margin of that axis alone had to hold the hit.
L = 5e-5
THIN = [((100, 0, -1, 101, 0, 1, 100.5, 6e-17, 1), (0, 0, .25, 1, 0, 0)),
        ((1, -1e-20, -1, 1, 1e-20, -1, 1, 0, 1), (0, 0, 0, 1, 0, 0)),
        ((1, -1e-10, -1, 1, 1e-10, -1, 1, 0, 1), (0, 0, 0, 2e-9, 0, 0)),
        ((0, 0, -L, 0, L, L, 0, 0, L), (-1, 0, 0, 2.0 ** -29, -0.0, 0)),
        ((0, 0, -1, 0, 1e-13, 1, 0, 0, 1), (-1, 0, 0, 1, -0.0, 0))]


def swap_yz(a):
    return np.asarray(a, F).reshape(-1, 3)[:, [0, 2, 1]].reshape(-1)


def test_thin_triangles(one_fma):
    tris, rays = [], []
    for t, r in THIN:
        for swapped in (False, True):
            for zero in (0.0, -0.0):
                tris.append(swap_yz(t) if swapped else t)
                r2 = swap_yz(r) if swapped else np.array(r, F)
                r2[3:][r2[3:] == 0] = zero
                rays.append(r2)
    check(one_fma, tris, rays)


def squeezed(rng, n):
    """Triangles squeezed by 1 to 1e-20 on the y and z axes, about 0 or not, and rays with d_y, d_z or both 0
    through a point of them, of lengths 2^-28 to 2^28."""
    v = rng.uniform(-1, 1, (n, 3, 3)) * 10.0 ** rng.uniform(-20, 2, (n, 1, 3))
    v[:, :, 0] = rng.uniform(-1, 1, (n, 3))
    v += np.where(rng.random((n, 1, 3)) < .3, rng.uniform(-5, 5, (n, 1, 3)), 0)
    v = v.astype(F).astype(np.float64)
    w = rng.dirichlet((1, 1, 1), n)[:, :, None]
    at = np.where(rng.random((n, 1)) < .7, (v * w).sum(1), v[:, 0])  # inside, or a vertex
    d = rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-3, 0, (n, 3))
    d[:, 0] = np.where(np.abs(d[:, 0]) < .05, .5, d[:, 0])
    zero = rng.integers(1, 4, n)
    d[zero & 1 == 1, 1] = 0
    d[zero & 2 == 2, 2] = 0
    o = at - d * rng.uniform(.01, 100, (n, 1))
    for k in (1, 2):
        o[d[:, k] == 0, k] = at[d[:, k] == 0, k]
    d = d * 2.0 ** rng.uniform(-20, 20, (n, 1))
    d = np.where(d == 0, np.where(rng.random((n, 3)) < .5, 0.0, -0.0), d)
    return v.reshape(n, 9).astype(F), np.concatenate([o, d], 1).astype(F)


def test_squeezed_triangles(one_fma):
    check(one_fma, *squeezed(np.random.default_rng(1), 20000))


def huge_directions(rng, n):
    """Rays of lengths 1e8 to 1e36 at triangles of 1e-32 to 1: t from ordinary to denormal."""
    size = 10.0 ** rng.uniform(-32, 0, (n, 1))
    v = (rng.uniform(-1, 1, (n, 9)) * size).astype(F)
    w = rng.dirichlet((1, 1, 1), n)[:, :, None]
    at = (v.reshape(n, 3, 3).astype(np.float64) * w).sum(1)
    d = rng.normal(size=(n, 3))
    d[rng.random(n) < .2, 1] = 0
    d[rng.random(n) < .2, 2] = 0
    o = at - d * size * 10.0 ** rng.uniform(-2, 2, (n, 1))
    return v, np.concatenate([o, d * 10.0 ** rng.uniform(8, 36, (n, 1))], 1).astype(F)


def test_huge_directions(one_fma):
    check(one_fma, *huge_directions(np.random.default_rng(3), 20000), exact=True)


def test_ordinary_rays_stay_fast(one_fma):
    """Parallel rays and the centre lines of a camera over a scene of ordinary proportions take the
    one-fma test, but for those with the coordinate 0 itself on the zero axis."""
    rng = np.random.default_rng(2)
    rays = rng.uniform(-2, 2, (4000, 6)).astype(F)
    rays[np.arange(4000) % 2 == 0, 4] = 0
    rays[np.arange(4000) % 3 == 0, 5] = 0
    assert one_fma(rays, np.full(4000, 30, F)).all()
    rays[:, 3:] *= 1000
    assert one_fma(rays, np.full(4000, 30, F)).all()
    rays[:, 3] = 0
    assert not one_fma(rays, np.full(4000, 30, F)).any()
