"""Timed cases of the ray-traversal library, through its public entry points.

What a user of the library has it do: trace ray sets against a resident tree (closest
hit and any hit, single rays and 64-ray packets, both triangle tests), trace frames of
several ray batches in one launch, animate a mesh and trace the refitted or updated tree,
build a tree on the device, generate and shade the rays of an image, and serve render
requests. Meshes are the library's two workload kinds at the sizes of its configurations
and between them: a triangle soup and a value-noise heightfield.

listed() names the cases, draw() gives others of the same ranges, prepare() makes the
inputs and handles of one, run() is one pass, work() what a pass cannot do without, and
exact() the hits of a small set in 64 bits.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from rfmanta_amd import _lib as L
from rfmanta_amd import api, scenes

MAXT = 1.0e19
T_EPSILON = 1.0e-4


def listed() -> list:
    return [
        # The smallest call: one 64x64 preview image of a 10,000-triangle mesh.
        {"name": "trace small", "do": "trace", "mesh": "soup", "tris": 10_000, "prim": "ks",
         "rays": "camera", "n": 4_096, "packet": 1},
        # Primary rays of a 1080p image over the 1M-triangle terrain.
        {"name": "trace primary", "do": "trace", "mesh": "heightfield", "tris": 997_002,
         "prim": "ks", "rays": "camera", "n": 2_073_600, "packet": 1},
        # The incoherent diffuse bounces of such an image, a ragged count.
        {"name": "trace bounce", "do": "trace", "mesh": "heightfield", "tris": 997_002,
         "prim": "ks", "rays": "bounce", "n": 1_000_003, "packet": 1},
        # Its shadow rays (any hit), with the other triangle test.
        {"name": "trace shadow wald", "do": "trace", "mesh": "heightfield", "tris": 997_002,
         "prim": "wald", "rays": "shadow", "n": 2_073_600, "packet": 1},
        # The reference's own 64-ray packets over a 1080p image.
        {"name": "trace packets", "do": "trace", "mesh": "heightfield", "tris": 997_002,
         "prim": "ks", "rays": "camera", "n": 2_073_600, "packet": 64},
        # The headline frame: primary and bounce batch in one launch, pinned configuration.
        {"name": "frame primary bounce", "do": "frame", "mesh": "heightfield", "tris": 997_002,
         "prim": "ks", "batches": 2, "n": 4_147_200, "launch": "pinned"},
        # Uneven batches of all three ray kinds in one launch, default configuration.
        {"name": "frame mixed", "do": "frame", "mesh": "soup", "tris": 300_000, "prim": "ks",
         "batches": 12, "n": 3_000_000, "launch": "default"},
        # An animated 8M-triangle terrain, bounds-only refit, 1080p primary rays.
        {"name": "refit frame", "do": "animate", "mesh": "heightfield", "tris": 7_990_002,
         "prim": "ks", "update": "refit", "n": 2_073_600},
        # The same with the reference's update (tree rotations and leaf splits).
        {"name": "update frame", "do": "animate", "mesh": "heightfield", "tris": 7_990_002,
         "prim": "ks", "update": "rotate", "n": 2_073_600},
        # A new tree on the device for 1M triangles, then the first image over it.
        {"name": "build", "do": "build", "mesh": "heightfield", "tris": 997_002, "prim": "ks",
         "n": 786_432},
        # One image from camera to shading inputs: camera rays, hits, shadow and bounce rays
        # and their hits, positions, normals and texture coordinates.
        {"name": "image", "do": "image", "mesh": "soup", "tris": 200_000, "prim": "ks",
         "xres": 1024, "yres": 768, "spp": 1},
        # Four render requests with shadows and bounces, results in host memory.
        {"name": "serve", "do": "serve", "mesh": "heightfield", "tris": 997_002, "prim": "ks",
         "requests": 4, "xres": 512, "yres": 512},
    ]


def draw(rng) -> dict:
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    do = rng.choice(["trace", "trace", "trace", "frame", "animate", "build", "image", "serve"])
    c = {"do": do, "mesh": rng.choice(["soup", "heightfield"]), "tris": log(1_000, 1_000_000),
         "prim": rng.choice(["ks", "ks", "wald"])}
    if do == "trace":
        c["rays"] = rng.choice(["camera", "bounce", "shadow", "random"])
        c["n"] = log(1_000, 2_000_000) | 1
        c["packet"] = rng.choice([1, 1, 1, 64])
        if c["packet"] > 1 and c["rays"] != "camera":
            c["n"] = min(c["n"], 500_001)
    elif do == "frame":
        c["batches"] = rng.randint(2, 12)
        c["n"] = log(100_000, 3_000_000)
        c["launch"] = rng.choice(["pinned", "default"])
    elif do == "animate":
        c["update"] = rng.choice(["refit", "rotate"])
        c["tris"] = log(10_000, 4_000_000)
        c["n"] = log(10_000, 2_000_000)
    elif do == "build":
        c["n"] = log(10_000, 1_000_000)
    elif do == "image":
        c["xres"], c["yres"] = 8 * rng.randint(16, 160), 8 * rng.randint(16, 100)
        c["spp"] = rng.randint(1, 2)
    else:
        c["requests"] = rng.randint(1, 4)
        c["xres"], c["yres"] = 8 * rng.randint(16, 64), 8 * rng.randint(16, 64)
    return c


# ---- meshes ------------------------------------------------------------------------------


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float32)


def _grid(tris: int) -> tuple:
    """Vertex grid of a heightfield of about `tris` triangles (2:1; 4:1 above 2M)."""
    a = 2.0 if tris < 2_000_000 else 4.0
    nz = max(2, int(round(math.sqrt(tris / (2 * a)))) + 1)
    nx = max(2, int(round(tris / (2 * (nz - 1)))) + 1)
    return nx, nz


def _soup_half(tris: int) -> float:
    return max(1.0, 4.0 * (tris / 8.0e6) ** (1.0 / 3.0))


def _mesh(case: dict, g) -> tuple:
    tris = case["tris"]
    if case["mesh"] == "soup":
        c = (2 * _rand(g, tris, 1, 3) - 1) * _soup_half(tris)
        e = 0.02 * torch.randn(tris, 3, 3, generator=g, device="cuda", dtype=torch.float32)
        v = (c + e).reshape(-1, 3)
        idx = torch.arange(3 * tris, device="cuda", dtype=torch.int32).reshape(tris, 3)
        return v.cpu().numpy(), idx.cpu().numpy().view(np.uint32)
    nx, nz = _grid(tris)
    half = (nz - 1) / (nx - 1)
    x = torch.linspace(-1, 1, nx, device="cuda")
    z = torch.linspace(-half, half, nz, device="cuda")
    h = torch.zeros(nz, nx, device="cuda")
    norm = 0.0
    for o in range(6):  # value-noise fBm, amplitude 0.2
        f = 4.0 * 2**o
        sx, sz = (x + 1) * 0.5 * f, (z + half) * 0.5 * f
        ix, iz = sx.floor().long(), sz.floor().long()
        lat = 2 * _rand(g, int(iz.max()) + 2, int(ix.max()) + 2) - 1
        fx, fz = sx - ix, sz - iz
        wx, wz = fx * fx * (3 - 2 * fx), (fz * fz * (3 - 2 * fz))[:, None]
        rows0, rows1 = lat[iz], lat[iz + 1]
        a = rows0[:, ix] + (rows0[:, ix + 1] - rows0[:, ix]) * wx
        b = rows1[:, ix] + (rows1[:, ix + 1] - rows1[:, ix]) * wx
        h += 0.5**o * (a + (b - a) * wz)
        norm += 0.5**o
    v = torch.stack([x.expand(nz, nx), 0.2 * h / norm, z[:, None].expand(nz, nx)], -1)
    j = torch.arange(nz - 1, device="cuda", dtype=torch.int32)[:, None]
    i = torch.arange(nx - 1, device="cuda", dtype=torch.int32)[None]
    v00 = (j * nx + i).reshape(-1)
    idx = torch.stack([v00, v00 + 1, v00 + nx + 1, v00, v00 + nx + 1, v00 + nx], -1)
    return (v.reshape(-1, 3).cpu().numpy(),
            idx.reshape(-1, 3).contiguous().cpu().numpy().view(np.uint32))


# ---- rays --------------------------------------------------------------------------------


class _Array:
    """A torch tensor where the API keeps device arrays."""

    def __init__(self, t: torch.Tensor):
        self.t, self.ptr = t, t.data_ptr()


def _f32(n):
    return _Array(torch.zeros(n, device="cuda", dtype=torch.float32))


def _alloc_rays(n: int) -> api.DeviceRays:
    arrays = {k: _f32(n) for k in api.RAY_FIELDS}
    arrays["masked"] = _Array(torch.zeros(n, device="cuda", dtype=torch.uint8))
    return api.DeviceRays(n, arrays)


def _first(rays: api.DeviceRays, n: int) -> api.DeviceRays:
    return api.DeviceRays(n, {k: _Array(a.t[:n].contiguous()) for k, a in rays.arrays.items()})


def _alloc_hits(n: int, any_hit: bool = False) -> api.DeviceHits:
    arrays = {"prim": _Array(torch.zeros(n, device="cuda", dtype=torch.int32)), "t": _f32(n),
              "u": _f32(n), "v": _f32(n)}
    if any_hit:
        arrays["occluded"] = _Array(torch.zeros(n, device="cuda", dtype=torch.uint8))
    return api.DeviceHits(n, arrays)


def _out(hits: api.DeviceHits, any_hit: bool = False) -> dict:
    """The hit record: triangle, distance and barycentrics, and an any-hit ray's flag."""
    keys = ("prim", "t", "u", "v") + (("occluded",) if any_hit else ())
    return {k: hits.arrays[k].t for k in keys}


def _view(case: dict, r) -> tuple:
    """An eye outside the mesh and its light, moved a little by the seed."""
    az, el = r.uniform(0, 2 * math.pi), r.uniform(0.6, 0.9)
    d = 1.6 if case["mesh"] == "heightfield" else 2.7 * _soup_half(case["tris"])
    eye = (d * math.cos(el) * math.cos(az), d * math.sin(el), d * math.cos(el) * math.sin(az))
    return eye, (2.0 * d, 2.0 * d, -1.5 * d)


def _camera(eye, xres: int, yres: int, spp: int = 1, seed: int = 0):
    return api.camera(eye, (0.0, 0.0, 0.0), (0, 1, 0), 40.0, xres, yres, spp=spp, seed=seed)


def _camera_rays(eye, n: int) -> api.DeviceRays:
    """The first n rays of a 16:9 image of at least n pixels."""
    if n == 2_073_600:
        xres, yres = 1920, 1080
    else:
        yres = max(8, 8 * int(math.ceil(math.sqrt(n * 9 / 16) / 8)))
        xres = 8 * int(math.ceil(n / yres / 8))
    rays = _alloc_rays(xres * yres)
    api.gen_camera_rays(_camera(eye, xres, yres), rays)
    return rays if rays.n == n else _first(rays, n)


def _random_rays(case: dict, n: int, g) -> api.DeviceRays:
    """Origins in the mesh's box, directions uniform on the sphere."""
    half = 1.0 if case["mesh"] == "heightfield" else _soup_half(case["tris"])
    o = (2 * _rand(g, 3, n) - 1) * half
    d = torch.randn(3, n, generator=g, device="cuda", dtype=torch.float32)
    d = d / d.norm(dim=0, keepdim=True)
    rays = _alloc_rays(n)
    for k, v in zip(api.RAY_FIELDS, [*o, *d, torch.full((n,), MAXT, device="cuda")]):
        rays.arrays[k].t.copy_(v)
    return rays


def _rays(case: dict, kind: str, n: int, scene, eye, light, seed: int, g) -> api.DeviceRays:
    if kind == "random":
        return _random_rays(case, n, g)
    primary = _camera_rays(eye, n)
    if kind == "camera":
        return primary
    hits = _alloc_hits(n)
    scene.trace(primary, hits)
    out = _alloc_rays(n)
    if kind == "bounce":
        api.gen_bounce_rays(scene, primary, hits, seed, out)
    else:
        api.gen_shadow_rays(scene, primary, hits, light, out)
    return out


# ---- cases -------------------------------------------------------------------------------


def prepare(case: dict, seed: int) -> dict:
    r = np.random.RandomState(seed % (1 << 32))
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    verts, idx = _mesh(case, g)
    scene = api.Scene(verts, idx)
    kind = L.MH_PRIM_WALD if case["prim"] == "wald" else L.MH_PRIM_KENSLER_SHIRLEY
    eye, light = _view(case, r)
    do = case["do"]
    state = {"do": do, "scene": scene, "kind": kind, "light": light, "seed": int(seed)}
    if do == "build":
        state["rays"] = _camera_rays(eye, case["n"])
        state["hits"] = _alloc_hits(case["n"])
        return state
    # The exact build on the host; above 2M triangles the device build.
    scene.build(prim_kind=kind, approximate=case["tris"] > 2_000_000)
    if do == "trace":
        any_hit = case["rays"] == "shadow"
        state["any"] = any_hit
        state["rays"] = _rays(case, case["rays"], case["n"], scene, eye, light, seed, g)
        state["hits"] = _alloc_hits(case["n"], any_hit)
        state["opts"] = api.trace_opts(packet_size=case["packet"]) if case["packet"] > 1 else None
    elif do == "frame":
        nb = case["batches"]
        if nb == 2:
            kinds, sizes = ["camera", "bounce"], [case["n"] // 2, case["n"] - case["n"] // 2]
        else:  # log-uniform sizes, 40% primary, 30% shadow, 30% bounce; the case's, not the seed's
            q = np.random.RandomState(nb + case["n"])
            w = np.exp(q.uniform(math.log(1e3), math.log(1e6), nb))
            sizes = [max(1, int(x)) for x in w / w.sum() * case["n"]]
            kinds = [str(k) for k in q.choice(["camera", "shadow", "bounce"], nb,
                                              p=[0.4, 0.3, 0.3])]
        batches = []
        for b, (k, n) in enumerate(zip(kinds, sizes)):
            e = eye if nb == 2 else _view(case, r)[0]
            batches.append((_rays(case, k, n, scene, e, light, seed + b, g),
                            _alloc_hits(n, k == "shadow"), k == "shadow"))
        state["batches"] = batches
        state["frame"] = api.Frame(scene, batches)
        if case["launch"] == "pinned":
            state["frame"].set_config(scenes.C1_LAUNCH)
    elif do == "animate":
        state["step"] = scene.refit if case["update"] == "refit" else scene.update
        state["phase"] = float(r.uniform(0, 2 * math.pi))
        state["rays"] = _camera_rays(eye, case["n"])
        state["hits"] = _alloc_hits(case["n"])
    elif do == "image":
        cam = _camera(eye, case["xres"], case["yres"], case["spp"], int(seed))
        n = case["xres"] * case["yres"] * case["spp"]
        state["camera"] = cam
        for k in ("primary", "shadow", "bounce"):
            state[k] = _alloc_rays(n)
            state[k + "_hits"] = _alloc_hits(n, k == "shadow")
        state["surface"] = [torch.zeros(n, device="cuda") for _ in range(12)]
        state["shading"] = L.Shading(*[a.data_ptr() for a in state["surface"]])
    else:
        state["server"] = api.Server([scene], shadows=True, bounces=True, light=light)
        state["cameras"] = [_camera(_view(case, r)[0], case["xres"], case["yres"], 1, seed + k)
                            for k in range(case["requests"])]
    return state


def run(state: dict):
    do, scene = state["do"], state["scene"]
    if do == "trace":
        scene.trace(state["rays"], state["hits"], state["any"], state["opts"])
        return _out(state["hits"], state["any"])
    if do == "frame":
        state["frame"].launch()
        return [_out(h, any_hit) for _, h, any_hit in state["batches"]]
    if do == "animate":  # the next frame of the animation
        state["phase"] += 0.1
        scene.displace_sine(0.01, 4.0, state["phase"])
        state["step"]()
        scene.trace(state["rays"], state["hits"])
        return _out(state["hits"])
    if do == "build":
        scene.build(prim_kind=state["kind"], approximate=True)
        scene.trace(state["rays"], state["hits"])
        stats = scene.stats()
        return {**_out(state["hits"]), "nodes": stats["nodes"], "depth": stats["depth"]}
    if do == "image":
        primary, hits = state["primary"], state["primary_hits"]
        api.gen_camera_rays(state["camera"], primary)
        scene.trace(primary, hits)
        api.gen_shadow_rays(scene, primary, hits, state["light"], state["shadow"])
        scene.trace(state["shadow"], state["shadow_hits"], any_hit=True)
        api.gen_bounce_rays(scene, primary, hits, state["seed"], state["bounce"])
        scene.trace(state["bounce"], state["bounce_hits"])
        r, h = primary.struct(), hits.struct()
        L.check(L.load().mh_shade(scene.h, r, h, primary.n, state["shading"], None))
        return {"hits": _out(hits), "shadow": _out(state["shadow_hits"], True),
                "bounce": _out(state["bounce_hits"]), "surface": state["surface"],
                "shadow rays": [state["shadow"].arrays[k].t for k in ("ox", "oy", "oz")],
                "bounce rays": [state["bounce"].arrays[k].t for k in ("dx", "dy", "dz")]}
    server = state["server"]
    ids = [server.submit(0, cam) for cam in state["cameras"]]
    done = [server.wait(i) for i in ids]
    return [{k: d[k] for k in ("prim", "t", "occluded", "bounce_prim", "bounce_t")} for d in done]


def work(case: dict) -> dict:
    """Rays in and hits out once, 44 bytes a ray; per ray about 2 log2(T) box tests of 25
    operations and 3 triangle tests of 45. An update reads each triangle's indices and
    vertices and writes its record (96 bytes) and two 32-byte tree records; a build also
    reads and writes what it sorts, once."""
    t, do = case["tris"], case["do"]
    n = case["n"] if "n" in case else case["xres"] * case["yres"]
    if do == "image":
        n *= 3 * case["spp"]
    if do == "serve":
        n *= 3 * case["requests"]
    b = 44.0 * n
    f = n * (25.0 * 2.0 * math.log2(t) + 3 * 45.0)
    if do in ("animate", "build"):
        b += t * (96.0 + 64.0)
        f += t * 30.0
    if do == "build":
        b += t * 96.0
        f += t * 40.0 * math.log2(t)
    return {"bytes": b, "flops": f}


def exact(case: dict, seed: int):
    """Closest hits of a small single-ray set by testing every triangle in 64 bits (the
    nearest intersection beyond T_EPSILON; triangle ids are left out)."""
    if (case["do"] != "trace" or case["rays"] == "shadow" or case["n"] * case["tris"] > 10**8
            or case["mesh"] != "soup"):
        return None
    state = prepare(case, seed)
    v = torch.from_numpy(state["scene"].verts).cuda().double()
    tri = v[torch.from_numpy(state["scene"].idx.astype(np.int64)).cuda()]
    p0, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    a = {k: x.t.double() for k, x in state["rays"].arrays.items() if k != "masked"}
    masked = state["rays"].arrays["masked"].t.bool()
    o = torch.stack([a["ox"], a["oy"], a["oz"]], 1)
    d = torch.stack([a["dx"], a["dy"], a["dz"]], 1)
    n = torch.linalg.cross(e1, e2)
    out = {k: torch.zeros(len(o), device="cuda", dtype=torch.float64) for k in ("t", "u", "v")}
    step = max(1, 4_000_000 // len(p0))
    for s in range(0, len(o), step):
        oo, dd = o[s:s + step, None], d[s:s + step, None]
        g = p0[None] - oo
        det = (dd * n[None]).sum(-1)
        t = (g * n[None]).sum(-1) / det
        w = oo + t[..., None] * dd - p0[None]
        nn = (n * n).sum(-1)[None]
        u = (torch.linalg.cross(w, e2[None].expand_as(w)) * n[None]).sum(-1) / nn
        q = (torch.linalg.cross(e1[None].expand_as(w), w) * n[None]).sum(-1) / nn
        ok = (t > T_EPSILON) & (t < a["tmax"][s:s + step, None]) & (u >= 0) & (q >= 0) & (u + q <= 1)
        best, at = torch.where(ok, t, torch.inf).min(1)
        hit = torch.isfinite(best) & ~masked[s:s + step]
        rows = torch.arange(len(at), device="cuda")
        miss = torch.where(masked[s:s + step], -a["tmax"].new_tensor(np.float32(MAXT)),
                           a["tmax"][s:s + step])
        out["t"][s:s + step] = torch.where(hit, best, miss)
        out["u"][s:s + step] = torch.where(hit, u[rows, at], 0.0)
        out["v"][s:s + step] = torch.where(hit, q[rows, at], 0.0)
    return {"prim": None, **out}
