"""Timed cases of the nearest-hit backend, each one pass through the public entry points.

The scenes are the repository's own (room, displaced icosphere, the closed 5,120-triangle stand-in
for the validation mesh, random soups, the 64-scene batch), moved and reordered from the seed; the
rays are drawn from the seed. Records are returned field by field as views of the record buffer.
"""
import functools
import math
import random

import numpy as np
import torch

import portablert_amd as prt
from portablert_amd import scenes

ALL = prt.mask_of(prt.ALL_TAGS)
T_ID = prt.T | prt.PRIMITIVE_ID
LARGEST_RAYS = 8388608


def listed():
    return [
        # one ray through the host call: mouse picking, a line-of-sight query, the reference's
        # single-ray examples; latency only
        {"name": "pick", "kind": "host", "scene": "blob", "tris": 5120, "rays": 1, "mask": ALL},
        # a small animated mesh: rebuilt every frame and seen through a 256 x 256 camera, everything
        # in host memory, all record fields (the reference's set_tris + nearest_hits loop)
        {"name": "frame", "kind": "build", "scene": "blob", "tris": 5120, "rays": 65536, "mask": ALL, "host": True},
        # a large static scene loaded from device memory, with a first batch of queries
        {"name": "build_room", "kind": "build", "scene": "room", "tris": 262144, "rays": 65536, "mask": T_ID,
         "host": False},
        # the largest scenes: an odd number of triangles above a million
        {"name": "build_large", "kind": "build", "scene": "soup", "tris": 1500001, "rays": 65536, "mask": T_ID,
         "host": False},
        # moving geometry of fixed topology: boxes updated and queried every step
        {"name": "refit_room", "kind": "refit", "scene": "room", "tris": 262144, "rays": 65536, "mask": T_ID},
        # a full-HD frame of primary rays, every record field (shading)
        {"name": "camera", "kind": "trace", "scene": "sphere", "tris": 81920, "rays": 2073600, "mask": ALL,
         "node_format": 1, "cull": 1, "leaf_test": 0},
        # an orthographic depth map from above (height fields, probe grids, picking along an axis):
        # parallel rays with two zero direction components
        {"name": "ortho", "kind": "trace", "scene": "room", "tris": 262144, "rays": 262144, "mask": T_ID,
         "node_format": 1, "cull": 1, "leaf_test": 0, "view": "ortho", "axis": 1},
        # the headline workload: 8,388,608 incoherent rays in the room, device resident
        {"name": "rays_room", "kind": "trace", "scene": "room", "tris": 262144, "rays": LARGEST_RAYS, "mask": T_ID,
         "node_format": 1, "cull": 1, "leaf_test": 0},
        # many rays from and to host vectors, the reference's only call form
        {"name": "host_room", "kind": "host", "scene": "room", "tris": 262144, "rays": 4194304, "mask": T_ID},
        # 64 scenes rebuilt and traced per step by one captured graph
        {"name": "batch", "kind": "batch", "scenes": 64, "counts": -1, "mask": T_ID, "graph": True},
        # learned seeding: network inference and the seeded traversal
        {"name": "learned", "kind": "learned", "scene": "room", "tris": 262144, "rays": 1048576, "mask": T_ID},
        # training of the seeding network: labels and 8 optimiser steps
        {"name": "train", "kind": "train", "scene": "room", "tris": 262144, "rays": 65536, "batch": 8192},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _scene(rng, most=1500000):
    kind = rng.choice(["blob", "sphere", "room", "soup"])
    tris = {"blob": 5120, "sphere": 81920, "room": 262144}.get(kind)
    return {"scene": kind, "tris": tris or _log_int(rng, 12, most)}


def draw(rng):
    kind = rng.choice(["host", "build", "refit", "trace", "trace", "batch", "learned", "train"])
    mask = rng.choice([T_ID, ALL, prt.T, prt.VALID, T_ID | prt.P])
    if kind == "host":
        return {"kind": kind, **_scene(rng), "rays": _log_int(rng, 1, 4194304), "mask": mask}
    if kind == "build":
        return {"kind": kind, **_scene(rng), "rays": _log_int(rng, 256, 65536), "mask": mask,
                "host": rng.random() < 0.5}
    if kind == "refit":
        return {"kind": kind, **_scene(rng), "rays": _log_int(rng, 256, 65536), "mask": mask}
    if kind == "trace":
        return {"kind": kind, **_scene(rng), "rays": _log_int(rng, 64, 4194304), "mask": mask,
                "node_format": rng.choice([1, 1, 1, 0]), "cull": rng.choice([1, 1, 0]), "leaf_test": rng.choice([0, 0, 1]),
                **({"view": "ortho", "axis": rng.randrange(3)} if rng.random() < 0.25 else {})}
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(2, 40), "counts": rng.randrange(1 << 20), "mask": T_ID,
                "graph": rng.random() < 0.5}
    if kind == "learned":
        return {"kind": kind, **_scene(rng, 300000), "rays": _log_int(rng, 1024, 1048576), "mask": mask}
    return {"kind": kind, **_scene(rng, 300000), "rays": 32 * _log_int(rng, 256, 2048),
            "batch": 32 * _log_int(rng, 32, 256)}


# ------------------------------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=None)
def _stream():
    """The program's one stream."""
    return torch.cuda.Stream()


@functools.lru_cache(maxsize=None)
def _mesh(kind):
    return scenes.scene({"blob": scenes.BUNNY, "sphere": scenes.SPHERE, "room": scenes.ROOM}[kind])


def _gen(seed, k):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + k) % (1 << 62))
    return g


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda")


def _soup(g, n, size):
    centre = 2.0 * _uniform(g, n, 1, 3) - 1.0
    return (centre + size * (2.0 * _uniform(g, n, 3, 3) - 1.0)).reshape(n, 9).contiguous()


def _triangles(case, seed):
    """Device triangles [n][9] and the scene's bounds (lo, hi) as two lists of 3."""
    g = _gen(seed, 1)
    n = case["tris"]
    if case["scene"] == "soup":
        return _soup(g, n, 0.05 * min(4.0, (16384.0 / n) ** (1.0 / 3.0)))
    v = torch.from_numpy(_mesh(case["scene"])).cuda().reshape(n, 3, 3)
    if case["scene"] == "room":  # stretched along its axes: walls and boxes stay in axis planes
        v = v * (0.9 + 0.2 * _uniform(g, 3)) + (2.0 * _uniform(g, 3) - 1.0)
    else:  # turned about a random axis (every copy of a shared vertex by the same operations)
        q = torch.randn(4, generator=g, device="cuda", dtype=torch.float64)
        w, x, y, z = (q / q.norm()).tolist()
        r = [[1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)],
             [2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)],
             [2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)]]
        d = v.double()
        c = d.reshape(-1, 3).mean(0)
        d = d - c
        v = torch.stack([d[..., 0] * r[k][0] + d[..., 1] * r[k][1] + d[..., 2] * r[k][2] for k in range(3)], -1)
        v = (v + c).float()
    return v.reshape(n, 9)[torch.randperm(n, generator=g, device="cuda")].contiguous()


def _directions(g, n):
    """Uniform on the sphere, in 64 bits and rounded once, as the repository's ray sets."""
    z = 2.0 * torch.rand(n, generator=g, device="cuda", dtype=torch.float64) - 1.0
    phi = 2.0 * math.pi * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    s = torch.sqrt(1.0 - z * z)
    return torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], 1).float()


def _rays(case, tris, seed, n):
    """Device rays [n][6]: a pinhole camera on the meshes, incoherent rays in rooms, soups and
    where the watertight test is asked for; "ortho": parallel rays along an axis."""
    g = _gen(seed, 2)
    v = tris.reshape(-1, 3)
    lo, hi = v.min(0).values, v.max(0).values
    if case.get("view") == "ortho":
        axis = case["axis"]
        w = max(1, int(round(math.sqrt(n))))
        i = torch.arange(n, device="cuda")
        px = torch.stack([i % w, torch.div(i, w, rounding_mode="floor")], 1).float()
        rays = torch.zeros(n, 6, device="cuda")
        a, b = [k for k in range(3) if k != axis]
        at = (px + _uniform(g, 2)) / w  # a pixel grid over the scene, moved by part of a pixel
        rays[:, a] = lo[a] + (hi - lo)[a] * at[:, 0]
        rays[:, b] = lo[b] + (hi - lo)[b] * at[:, 1]
        rays[:, axis] = lo[axis] - 0.1 * (hi - lo)[axis]
        rays[:, 3 + axis] = 1.0
        return rays
    if case["scene"] in ("room", "soup") or case.get("leaf_test") == 1:
        o = lo + (hi - lo) * _uniform(g, n, 3)
        return torch.cat([o, _directions(g, n)], 1).contiguous()
    w = max(1, int(round(math.sqrt(n * 16.0 / 9.0))))
    h = -(-n // w)
    i = torch.arange(n, device="cuda")
    x, y = (i % w).float(), torch.div(i, w, rounding_mode="floor").float()
    shift = _uniform(g, 2)
    tan = math.tan(math.pi / 6.0)
    d = torch.stack([(2.0 * (x + shift[0]) / w - 1.0) * tan * (w / h), (1.0 - 2.0 * (y + shift[1]) / h) * tan,
                     torch.ones_like(x)], 1)
    if n == 1:
        d[:, :2] = 0.1 * (shift - 0.5)
    centre = (lo + hi) / 2
    eye = centre - torch.tensor([0.0, 0.0, 1.0], device="cuda") * (1.4 + 0.2 * _uniform(g, 1)) * (hi - lo).max()
    return torch.cat([eye.expand(n, 3), d / d.norm(dim=1, keepdim=True)], 1).contiguous()


def _batch_counts(case):
    if case["counts"] < 0:  # the repository's batch: 64 scenes, 2,516,661 triangles, 24,428,377 rays
        s = range(scenes.n_scenes(scenes.BATCH))
        return ([int(scenes.lib().prt_scene_tris(scenes.BATCH, k)) for k in s],
                [int(scenes.n_rays(scenes.BATCH, k)) for k in s])
    r = random.Random(case["counts"])
    most_t, most_r = r.choice([2e3, 2e4, 1e5]), r.choice([1e4, 1e5, 5e5])
    return ([_log_int(r, 1e2, most_t) for _ in range(case["scenes"])],
            [_log_int(r, 1e3, most_r) for _ in range(case["scenes"])])


def _records(mask, n):
    """A record buffer of n records as 32-bit words (every record is a whole number of them)."""
    return torch.empty(n, prt.layout(mask)[0] // 4, dtype=torch.int32, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        tc, rc = _batch_counts(case)
        g = _gen(seed, 3)
        tris = _soup(g, sum(tc), 0.05)
        n = sum(rc)
        rays = torch.empty(n, 6, device="cuda")
        rays[:, :3] = 2.0 * _uniform(g, n, 3) - 1.0
        rays[:, 3:] = _directions(g, n)
        ctx = prt.Context(0)
        out = _records(case["mask"], n)
        torch.cuda.synchronize()
        b = prt.Batch(ctx, tc, rc, case["mask"])
        b.run(tris.data_ptr(), rays.data_ptr(), out.data_ptr())
        b.check()
        if case["graph"]:
            b.capture(tris.data_ptr(), rays.data_ptr(), out.data_ptr())
        return {"case": case, "ctx": ctx, "batch": b, "tris": tris, "rays": rays, "out": out}
    tris = _triangles(case, seed)
    n = case["rays"]
    ctx = prt.Context(0)
    s = {"case": case, "ctx": ctx, "n_tris": len(tris)}
    for opt in ("node_format", "cull", "leaf_test"):
        if opt in case:
            ctx.set_option(opt, case[opt])
    if kind == "build" and case["host"]:
        s["tris"], s["rays"] = tris.cpu().numpy(), _rays(case, tris, seed, n).cpu().numpy()
        return s
    if kind == "host":
        ctx.set_tris(tris.cpu().numpy())
        s["rays"] = _rays(case, tris, seed, n).cpu().numpy()
        return s
    s["rays"] = _rays(case, tris, seed, n)
    if kind != "train":
        s["out"] = _records(case["mask"], n)
    torch.cuda.synchronize()  # the library reads the triangles on its own stream
    if kind == "build":
        s["tris"] = tris
        return s
    ctx.set_tris_device(tris.data_ptr(), len(tris))
    if kind == "refit":
        v = tris.reshape(-1, 3)
        size = 1e-3 * float((v.max(0).values - v.min(0).values).max())
        s["tris"] = (tris + size * (2.0 * _uniform(_gen(seed, 4), *tris.shape) - 1.0)).contiguous()
    elif kind in ("learned", "train"):
        prt.learned_setup(ctx, seed=1 + seed % 1000)
        if kind == "learned":
            some = _rays(case, tris, seed + 7, 524288)
            torch.cuda.synchronize()
            prt.learned_train(ctx, some.data_ptr(), len(some), epochs=1, batch=8192)
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------------------------- passes

def _fields(out, mask):
    """The record buffer's fields as views (the word of `valid` holds its byte and zero padding)."""
    _, off = prt.layout(mask)
    f = out.view(torch.float32)
    return {name: (out if name in ("primitive_id", "valid") else f)[:, o // 4]
            for name, o in zip(("u", "v", "t", "primitive_id", "valid", "px", "py", "pz"), off) if o >= 0}


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "host":
        hits = ctx.nearest_hits(s["rays"], case["mask"])
        return {k: hits[k] for k in hits.dtype.names}
    if kind == "build" and case["host"]:
        ctx.set_tris(s["tris"])
        hits = ctx.nearest_hits(s["rays"], case["mask"])
        return {k: hits[k] for k in hits.dtype.names}
    st = _stream().cuda_stream
    if kind == "batch":
        if case["graph"]:
            s["batch"].replay(st)
        else:
            s["batch"].run(s["tris"].data_ptr(), s["rays"].data_ptr(), s["out"].data_ptr(), st)
        return _fields(s["out"], case["mask"])
    rays = s["rays"]
    if kind == "train":
        prt.learned_train(ctx, rays.data_ptr(), len(rays), epochs=1, batch=case["batch"])
        return [prt.mlp_params(ctx, layer) for layer in range(4)]
    if kind == "build":
        ctx.set_tris_device(s["tris"].data_ptr(), s["n_tris"])
    elif kind == "refit":
        ctx.refit_device(s["tris"].data_ptr(), s["n_tris"])
    if kind == "learned":
        prt.nearest_hits_learned_device(ctx, rays.data_ptr(), len(rays), case["mask"], s["out"].data_ptr(), st)
    else:
        ctx.nearest_hits_device(rays.data_ptr(), len(rays), case["mask"], s["out"].data_ptr(), st)
    return _fields(s["out"], case["mask"])


def work(case):
    """Rays and triangles read once, records written once; the network's products where there is one."""
    params = sum(o * i for o, i in prt.LAYER_SHAPES)
    if case["kind"] == "batch":
        tc, rc = _batch_counts(case)
        return {"bytes": 36 * sum(tc) + (24 + prt.layout(case["mask"])[0]) * sum(rc), "flops": 0}
    if case["kind"] == "train":
        steps = case["rays"] // case["batch"]
        # per step: the weights and two moments read and written in 32 bits
        return {"bytes": 24 * case["rays"] + steps * 24 * params, "flops": 6 * params * steps * case["batch"]}
    b = 36 * case["tris"] + (24 + prt.layout(case["mask"])[0]) * case["rays"]
    return {"bytes": b, "flops": 2 * params * case["rays"] if case["kind"] == "learned" else 0}


# ---------------------------------------------------------------------------------- in 64 bits

def _nearest64(tris, rays):
    """Nearest hit of every ray over every triangle in 64 bits: the slab test on the triangle's own
    box, then Moller-Trumbore with inclusive bounds and no range check on t; equal t to the lowest
    index. Returns t (inf for a miss), u, v."""
    v = tris.double().reshape(-1, 3, 3)
    v0, e1, e2 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    lo, hi = v.min(1).values, v.max(1).values
    n = len(rays)
    t_all = torch.full((n,), math.inf, dtype=torch.float64, device=rays.device)
    u_all, v_all = torch.zeros_like(t_all), torch.zeros_like(t_all)

    def dot(a, b):
        return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]

    def cross(a, b):
        return a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]

    per = max(1, (1 << 25) // len(v0))
    for f in range(0, n, per):
        r = rays[f:f + per].double()
        o, d = [r[:, k:k + 1] for k in range(3)], [r[:, 3 + k:4 + k] for k in range(3)]
        near = far = None
        for k in range(3):
            a, b = (lo[:, k] - o[k]) / d[k], (hi[:, k] - o[k]) / d[k]
            near = torch.minimum(a, b) if near is None else torch.maximum(near, torch.minimum(a, b))
            far = torch.maximum(a, b) if far is None else torch.minimum(far, torch.maximum(a, b))
        ok = (far >= 0) & (near <= far * (1 + 1e-12 * torch.sign(far)))
        del near, far
        E1, E2 = [e1[:, k] for k in range(3)], [e2[:, k] for k in range(3)]
        p = cross(d, E2)
        det = dot(E1, p)
        s = [o[k] - v0[:, k] for k in range(3)]
        uu = dot(s, p) / det
        q = cross(s, E1)
        vv = dot(d, q) / det
        tt = dot(E2, q) / det
        ok &= (det != 0) & (uu >= 0) & (uu <= 1) & (vv >= 0) & (uu + vv <= 1)
        tt = torch.where(ok, tt, torch.full_like(tt, math.inf))
        best, at = tt.min(1)
        hit = torch.isfinite(best)
        t_all[f:f + per] = best
        u_all[f:f + per] = torch.where(hit, uu.gather(1, at[:, None])[:, 0], torch.zeros_like(best))
        v_all[f:f + per] = torch.where(hit, vv.gather(1, at[:, None])[:, 0], torch.zeros_like(best))
    return t_all, u_all, v_all


def exact(case, seed):
    if case["kind"] in ("batch", "learned", "train") or case["tris"] * case["rays"] > 6e10 or not case["mask"] & prt.T:
        return None
    s = prepare(case, seed)
    rays = torch.as_tensor(s["rays"]).cuda()
    tris = torch.as_tensor(s["tris"]).cuda() if "tris" in s else _triangles(case, seed)
    t, u, v = _nearest64(tris, rays)
    r = rays.double()
    got = {"t": t}
    if case["mask"] & prt.UV:
        got.update(u=u, v=v)
    if case["mask"] & prt.P:
        for k, name in enumerate(("px", "py", "pz")):
            got[name] = r[:, k] + t * r[:, 3 + k]
    for name, tag in (("primitive_id", prt.PRIMITIVE_ID), ("valid", prt.VALID)):
        if case["mask"] & tag:
            got[name] = None
    return got
