"""The work that a program using barney_amd has it do, as timed cases.

Six kinds, over the sizes that the benchmark, the tests and the demo scenes use:

  frame   render a frame of a resident world from scratch (reset, spp samples, read back): triangles and
          spheres, instanced tubes and cones, terrain under an HDRI map, structured, tet and mixed-cell volumes
  edit    set a volume's transfer function, then render a frame: a step of an interactive session
  trace   closest or any hit of a batch of rays that lie in device memory
  build   BVH builds over new geometry, then a first batch of rays through them
  serve   a burst of requests of mixed worlds, resolutions and sample counts through the request server

Scenes, cameras and rays come from the seed.  Every frame is summed in 2^-32 fixed point and every float
operation is pinned (no contraction, correctly rounded division and square root), so a pixel does not depend
on the order of the work and outputs are compared exactly.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import numpy as np
import torch

import barney_amd as bx
from barney_amd import abi, scenes

GPU = "cuda:0"
CHANNELS = {"color": abi.BNX_FB_COLOR, "srgb8": abi.BNX_FB_COLOR_SRGB8, "rgba8": abi.BNX_FB_COLOR_RGBA8,
            "depth": abi.BNX_FB_DEPTH, "prim": abi.BNX_FB_PRIMID, "inst": abi.BNX_FB_INSTID,
            "obj": abi.BNX_FB_OBJID, "normal": abi.BNX_FB_NORMAL}


def listed():
    return [
        # the smallest call: a thumbnail of a small scene, where launches and read-backs are most of the time
        dict(name="frame_thumbnail", kind="frame", scene="surface", size=3, spheres=200, w=96, h=96, spp=1,
             read="srgb8"),
        # the plain surface frame: icosphere and 1,000 spheres, one directional light
        dict(name="frame_surface", kind="frame", scene="surface", size=5, spheres=1000, w=512, h=512, spp=1,
             read="color"),
        # tubes, streamlines and arrows, each group placed many times by rotated instances, at an odd size,
        # with the channels that a compositor takes
        dict(name="frame_instances", kind="frame", scene="tubes", size=600, copies=27, w=641, h=363, spp=4,
             read="color,depth,prim,normal"),
        # the largest surface frame: millions of triangles and spheres, half of them glossy, HDRI light,
        # five generations
        dict(name="frame_terrain", kind="frame", scene="terrain", size=4096, spheres=4000000, w=1920, h=1080, spp=8,
             read="color"),
        # a small volume of odd sizes while its transfer function is being edited
        dict(name="edit_volume", kind="edit", scene="volume", size=97, w=333, h=217, spp=1, ratio=True,
             read="srgb8"),
        # the structured volume frame: 256^3 field, delta tracking, scattering
        dict(name="frame_volume", kind="frame", scene="volume", size=256, w=1024, h=1024, spp=16, ratio=False,
             read="color"),
        # a tetrahedral volume with an isosurface in it
        dict(name="frame_tets", kind="frame", scene="tets", size=160, w=1024, h=1024, spp=4, read="color"),
        # the same field on hexahedra, prisms, pyramids and tets
        dict(name="frame_cells", kind="frame", scene="cells", size=14, w=320, h=240, spp=2, read="color"),
        # picking and line-of-sight queries on a mid-sized scene
        dict(name="trace_closest", kind="trace", scene="surface", size=5, spheres=1000, rays=60001, any=False),
        # occlusion rays of a large scene
        dict(name="trace_any", kind="trace", scene="terrain", size=1025, spheres=100000, rays=1 << 20, any=True),
        # time-varying geometry: new triangles every step
        dict(name="build_mesh", kind="build", scene="terrain", size=725, spheres=50000, rays=65536),
        # a burst of requests
        dict(name="serve_burst", kind="serve", scene="mix", size=257, requests=24, top=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "edit", "trace", "trace", "build", "serve"])
    if kind == "frame":
        scene = rng.choice(["surface", "tubes", "terrain", "volume", "tets", "cells"])
        c = dict(kind=kind, scene=scene, read=rng.choice(["color", "srgb8", "rgba8", "color,depth,obj"]))
        w = _log(rng, 64, 1920)
        h = max(48, min(1080, int(w * rng.uniform(0.5, 1.0))))
        c.update(w=w, h=h, spp=_log(rng, 1, max(1, min(16, (16 << 20) // (w * h)))))
        if scene == "surface":
            c.update(size=rng.randint(1, 6), spheres=_log(rng, 10, 20000))
        elif scene == "tubes":
            c.update(size=_log(rng, 40, 4000), copies=rng.choice([1, 8, 27]))
        elif scene == "terrain":
            c.update(size=_log(rng, 33, 1500), spheres=_log(rng, 100, 500000), spp=min(c["spp"], 4))
        elif scene == "volume":
            c.update(size=_log(rng, 24, 256), ratio=rng.random() < 0.3)
        elif scene == "tets":
            c.update(size=_log(rng, 8, 80), spp=min(c["spp"], 2))
        else:
            c.update(size=rng.randint(4, 14), spp=1, w=min(w, 480), h=min(h, 360))
        return c
    if kind == "edit":
        return dict(kind=kind, scene="volume", size=_log(rng, 24, 200), w=_log(rng, 128, 900), h=_log(rng, 96, 700),
                    spp=_log(rng, 1, 4), ratio=rng.random() < 0.5, read="srgb8")
    if kind == "trace":
        scene = rng.choice(["surface", "tubes", "terrain"])
        c = dict(kind=kind, scene=scene, rays=_log(rng, 500, 2000000), any=rng.random() < 0.5)
        if scene == "surface":
            c.update(size=rng.randint(1, 6), spheres=_log(rng, 10, 20000))
        elif scene == "tubes":
            c.update(size=_log(rng, 40, 4000), copies=rng.choice([1, 8, 27]))
        else:
            c.update(size=_log(rng, 33, 1200), spheres=_log(rng, 100, 200000))
        return c
    if kind == "build":
        return dict(kind=kind, scene="terrain", size=_log(rng, 12, 1200), spheres=_log(rng, 30, 500000),
                    rays=_log(rng, 1000, 200000))
    return dict(kind=kind, scene="mix", size=_log(rng, 65, 400), requests=rng.randint(3, 24),
                top=rng.choice([256, 512, 1024]))


# ------------------------------------------------------------------ scenes
_device = None


def device():
    """the program's device: its stream, queues and captured loops serve every world"""
    global _device
    if _device is None:
        _device = bx.Device(0)
    return _device


def _gen(seed):
    return torch.Generator(device=GPU).manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=GPU)


def _light(radiance=1.0):
    return (-np.ones(3) / math.sqrt(3.0)).astype(np.float32), radiance, np.ones(3, np.float32)


def _orbit(seed, target, radius, fovy, lo=5.0, hi=50.0):
    r = np.random.default_rng(seed)
    az, el = r.uniform(0, 2 * math.pi), math.radians(r.uniform(lo, hi))
    p = np.asarray(target) + radius * np.array([math.cos(el) * math.sin(az), math.sin(el),
                                                math.cos(el) * math.cos(az)])
    return dict(position=tuple(p), direction=tuple(np.asarray(target) - p), up=(0.0, 1.0, 0.0), fovy=fovy)


def surface_scene(case, seed):
    """an icosphere among small spheres, one colour per primitive"""
    r = np.random.default_rng(seed)
    v, f = scenes.icosphere(case["size"])
    s = scenes.SurfaceScene()
    s.meshes.append(scenes.TriMesh(v, f, r.uniform(0.2, 0.8, (len(f), 3)).astype(np.float32), user_id=0))
    n = case["spheres"]
    s.spheres.append(scenes.SphereSet(r.uniform(-2, 2, (n, 3)).astype(np.float32),
                                      r.uniform(0.01, 0.05, n).astype(np.float32),
                                      r.uniform(0.2, 0.8, (n, 3)).astype(np.float32), user_id=1))
    s.dir_lights.append(_light())
    s.camera = _orbit(seed, (0.0, 0.0, 0.0), 5.0, 40.0, -30.0, 60.0)
    return s


def _heights(g, u, w, octaves=8):
    """value noise of 8 octaves at (u, w) in [0, 1]"""
    h = torch.zeros_like(u)
    for o in range(octaves):
        k = 4 << o
        lat = 2.0 * _rand(g, k + 1, k + 1) - 1.0
        x, z = u * k, w * k
        i, j = x.long().clamp_(max=k - 1), z.long().clamp_(max=k - 1)
        tx, tz = x - i, z - j
        tx = tx * tx * tx * (tx * (tx * 6 - 15) + 10)
        tz = tz * tz * tz * (tz * (tz * 6 - 15) + 10)
        a = lat[j, i] + (lat[j, i + 1] - lat[j, i]) * tx
        b = lat[j + 1, i] + (lat[j + 1, i + 1] - lat[j + 1, i]) * tx
        h += 0.12 * 0.5 ** o * (a + (b - a) * tz)
    return h


def terrain_scene(case, seed):
    """a heightfield with spheres lying on it, half of the primitives glossy, under an HDRI map"""
    n, ns, e = case["size"], case["spheres"], 16.0
    g = _gen(seed)
    line = torch.linspace(0.0, 1.0, n, device=GPU)
    w, u = torch.meshgrid(line, line, indexing="ij")
    su, sw, sr = _rand(g, ns), _rand(g, ns), 0.002 + 0.008 * _rand(g, ns)
    # one lattice for ground and spheres: the noise is drawn once, over both sets of points
    y = e * _heights(g, torch.cat([u.reshape(-1), su]), torch.cat([w.reshape(-1), sw]))
    verts = torch.stack([e * (2 * u.reshape(-1) - 1), y[:n * n], e * (2 * w.reshape(-1) - 1)], 1)
    centers = torch.stack([e * (2 * su - 1), y[n * n:] + sr, e * (2 * sw - 1)], 1)
    k = torch.arange(n - 1, device=GPU, dtype=torch.int32)
    i0 = (k[None, :] + n * k[:, None]).reshape(-1)
    tris = torch.stack([i0, i0 + n, i0 + 1, i0 + 1, i0 + n, i0 + n + 1], 1).reshape(-1, 3)
    tcol = 0.2 + 0.6 * _rand(g, len(tris), 3)
    glossy_t, glossy_s = _rand(g, len(tris)) < 0.5, _rand(g, ns) < 0.5
    scol = 0.2 + 0.6 * _rand(g, ns, 3)
    pbr = abi.pbr(metallic=0.0, roughness=0.2)
    host = lambda t: t.contiguous().cpu().numpy()  # noqa: E731
    s = scenes.SurfaceScene()
    vh = host(verts)
    for keep, mat, uid in ((~glossy_t, None, 0), (glossy_t, pbr, 1)):
        s.meshes.append(scenes.TriMesh(vh, host(tris[keep]), host(tcol[keep]), user_id=uid, material=mat))
    for keep, mat, uid in ((~glossy_s, None, 2), (glossy_s, pbr, 3)):
        s.spheres.append(scenes.SphereSet(host(centers[keep]), host(sr[keep]), host(scol[keep]), user_id=uid,
                                          material=mat))
    s.env = scenes.lobe_env_map(256, 128, seed=seed)
    s.max_generations = 5
    s.camera = _orbit(seed, (0.0, 0.0, 0.0), 9.0, 45.0, 15.0, 45.0)
    return s


def volume_scene(case, seed):
    """Gaussian blobs on a grid whose three sides differ a little"""
    n = case["size"]
    dims = (n, n, n) if n % 2 == 0 else (n, max(4, n - n // 5), max(4, n - n // 7))
    g = _gen(seed)
    f = torch.zeros(dims[2], dims[1], dims[0], device=GPU)
    c, s, a = _rand(g, 32, 3), 0.02 + 0.08 * _rand(g, 32), 0.5 + 0.5 * _rand(g, 32)
    ax = [torch.linspace(0.0, 1.0, d, device=GPU) for d in dims]
    for b in range(32):
        x, y, z = (torch.exp(-((ax[k] - c[b, k]) ** 2) / (2 * s[b] ** 2)) for k in range(3))
        f += a[b] * z[:, None, None] * y[None, :, None] * x[None, None, :]
    f = (f - f.min()) / (f.max() - f.min())
    v = scenes.StructuredVolumeScene(
        scalars=f.cpu().numpy(), grid_origin=(0.0, 0.0, 0.0), grid_spacing=tuple(1.0 / (d - 1) for d in dims),
        tf=scenes.ramp_tf(256, 0.8), tf_domain=(0.0, 1.0), base_density=50.0,
        cells_per_mc=max(1, -(-(n - 1) // 16)), dir_lights=[_light(2.5)])
    v.camera = _orbit(seed, (0.5, 0.5, 0.5), 2.7, 35.0)
    return v


def _umesh(seed, verts, scalars, tets, cells, mc):
    u = scenes.UMeshVolumeScene(vertices=verts, scalars=scalars, tets=tets, tf=scenes.ramp_tf(256, 0.8),
                                tf_domain=(float(scalars.min()), float(scalars.max())), base_density=50.0,
                                mc_dims=mc, cells=cells, dir_lights=[_light(2.5)])
    u.camera = _orbit(seed, (0.5, 0.5, 0.5), 2.7, 35.0)
    return u


def tets_scene(case, seed):
    """a jittered lattice of cubes, five tets each, with a noisy product of sines at the vertices"""
    n = case["size"]
    m, g = n + 1, _gen(seed)
    line = torch.arange(m, device=GPU)
    k, j, i = torch.meshgrid(line, line, line, indexing="ij")
    idx = torch.stack([i.reshape(-1), j.reshape(-1), k.reshape(-1)], 1)
    off = (2.0 * _rand(g, m ** 3, 3) - 1.0) * 0.2
    off[(idx == 0) | (idx == n)] = 0.0
    p = (idx + off) / n
    f = torch.sin(4 * p[:, 0]) * torch.cos(4 * p[:, 1]) * torch.sin(4 * p[:, 2])
    f += 0.05 * torch.randn(m ** 3, generator=g, device=GPU)
    line = torch.arange(n, device=GPU)
    k, j, i = (t.reshape(-1) for t in torch.meshgrid(line, line, line, indexing="ij"))

    def at(a, b, c):
        return (i + a) + m * ((j + b) + m * (k + c))

    v = {(a, b, c): at(a, b, c) for a in (0, 1) for b in (0, 1) for c in (0, 1)}
    tet = []
    for odd in (0, 1):
        # the middle tet joins four corners of which no two share an edge; cubes of odd index sum use the others
        mid = [c for c in v if (sum(c) & 1) == odd]
        own = [[v[c] for c in mid]]
        for c in v:
            if (sum(c) & 1) != odd:
                near = [d for d in mid if sum(abs(x - y) for x, y in zip(c, d)) == 1]
                own.append([v[c]] + [v[d] for d in near])
        tet.append(torch.stack([torch.stack(t, 1) for t in own], 1))
    tets = torch.where((((i + j + k) & 1) == 0)[:, None, None], tet[0], tet[1]).reshape(-1, 4)
    a, b, c, d = (p[tets[:, q]].double() for q in range(4))
    flip = ((torch.linalg.cross(b - a, c - a) * (d - a)).sum(1) < 0)
    tets[flip] = tets[flip][:, [0, 1, 3, 2]]
    return _umesh(seed, p.float().cpu().numpy(), f.float().cpu().numpy(), tets.int().cpu().numpy(), None, (32, 32, 32))


def cells_scene(case, seed):
    v, idx, offs, types = scenes.mixed_cells(case["size"], int(seed), jitter=0.15)
    p = v.astype(np.float64)
    f = (np.sin(4 * p[:, 0]) * np.cos(4 * p[:, 1]) * np.sin(4 * p[:, 2])).astype(np.float32)
    return _umesh(seed, v, f, np.zeros((0, 4), np.int32), (idx, offs, types), (8, 8, 8))


def _rotations(seed, copies):
    """affine transforms (12 floats, columns then origin) on a cubic raster, each turned and scaled its own way"""
    r, side = np.random.default_rng(seed + 1), round(copies ** (1 / 3))
    out = []
    for c in range(copies):
        q = r.normal(size=4)
        w, x, y, z = q / np.linalg.norm(q)
        m = np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                      [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                      [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]])
        at = np.array([c % side, (c // side) % side, c // (side * side)]) - (side - 1) / 2
        out.append(np.concatenate([(0.5 / side * m).T.reshape(-1), 2.2 / side * at]))
    return np.asarray(out, np.float32)


class World:
    """a world with everything that it keeps on the device, given back when it goes"""

    def __init__(self, case, seed):
        dev = self.dev = device()
        self.geoms, self.groups, self.vols, self.isos = [], [], [], []
        self.ambient, self.gens, kind = 1.0, 0, case["scene"]
        if kind in ("surface", "terrain"):
            sc = surface_scene(case, seed) if kind == "surface" else terrain_scene(case, seed)
            w = bx.SurfaceWorld(dev, sc)
            self.geoms, self.groups = w.sph + w.cyl + w.cap + w.cone + w.tri, w.groups
            self.insts, self.world, self.gens = w.insts, w.world, sc.max_generations
        elif kind == "tubes":
            n = case["size"]
            sc = scenes.SurfaceScene(cylinders=[scenes.sticks(n, seed)], capsules=[scenes.capsule_chains(n, seed)],
                                     cones=[scenes.cone_set(n // 2, seed)])
            cy, ca, co = sc.cylinders[0], sc.capsules[0], sc.cones[0]
            self.geoms = [bx.Geom.cylinders(dev, cy.vertices, cy.indices, cy.radii, cy.colors, user_id=4),
                          bx.Geom.capsules(dev, ca.vertices, ca.indices, ca.colors, user_id=5),
                          bx.Geom.cones(dev, co.vertices, co.radii, co.indices, co.colors, user_id=6)]
            self.groups = [bx.Group.geoms(dev, bx.USER, [g]).build() for g in self.geoms]
            x = _rotations(seed, case["copies"])
            self.insts = bx.Group.instances(dev, self.groups * len(x), None, np.repeat(x, 3, axis=0)).build()
            self.world = bx.World(dev, self.insts, [_light()])
            sc.camera = _orbit(seed, (0.0, 0.0, 0.0), 5.0, 40.0, -30.0, 60.0)
        else:
            sc = {"volume": volume_scene, "tets": tets_scene, "cells": cells_scene}[kind](case, seed)
            w = bx.VolumeWorld(dev, sc) if kind == "volume" else bx.UMeshWorld(dev, sc)
            self.insts, self.world, self.vols = w.insts, w.world, [w.volume]
            self.isos = [w.iso] if kind != "volume" else []
            self.ambient = 0.25
        c = sc.camera
        self.cam = bx.camera_perspective(c["position"], c["direction"], c["up"], c["fovy"])
        flags = abi.BNX_RENDER_RATIO_TRACKING if case.get("ratio") else 0
        self.rend = abi.renderer(bg=(0.0, 0.0, 0.0, 1.0), ambient=self.ambient, flags=flags, max_generations=self.gens)
        self.base = dict(c, target=tuple(np.add(c["position"], c["direction"])))

    def __del__(self):
        lib = bx.lib()
        lib.bnx_device_sync(self.dev.h)
        if hasattr(self, "world"):
            lib.bnx_world_destroy(self.world.h)
        for s in self.isos:
            lib.bnx_isosurface_destroy(s.h)
        for v in self.vols:
            lib.bnx_volume_destroy(v.h)
        for g in ([self.insts] if hasattr(self, "insts") else []) + self.groups:
            lib.bnx_group_destroy(g.h)
        for g in self.geoms:
            lib.bnx_geom_destroy(g.h)


def _rays(case, seed):
    """rays from a sphere around the scene (the terrain: from near its ground) towards it"""
    n, g = case["rays"], _gen(seed + 3)
    u = _rand(g, n, 6)
    r = torch.zeros(n, 8, device=GPU)
    if case["scene"] == "terrain":
        org = torch.stack([12 * (2 * u[:, 0] - 1), 0.5 + 2.0 * u[:, 1], 12 * (2 * u[:, 2] - 1)], 1)
        tgt = org + torch.stack([2 * u[:, 3] - 1, 0.6 - u[:, 4], 2 * u[:, 5] - 1], 1)
    else:
        z, phi = 1.0 - 2.0 * u[:, 0], 2 * math.pi * u[:, 1]
        q = torch.sqrt((1 - z * z).clamp_(min=0))
        org = 4.0 * torch.stack([q * torch.cos(phi), q * torch.sin(phi), z], 1)
        tgt = 1.5 * (2 * u[:, 2:5] - 1)
    d = tgt - org
    r[:, 0:3], r[:, 4:7], r[:, 7] = org, d / d.norm(dim=1, keepdim=True), 64.0
    return r


# ------------------------------------------------------------------ states
class State:
    def __del__(self):
        if hasattr(self, "server"):
            self.server.close()
        if hasattr(self, "frame"):
            self.frame.close()


def prepare(case, seed):
    st, kind = State(), case["kind"]
    st.case = case
    if kind == "serve":
        n, top, r = case["size"], case["top"], np.random.default_rng(seed)
        st.worlds = [World(dict(scene="surface", size=4, spheres=500), seed),
                     World(dict(scene="volume", size=min(128, n)), seed + 1),
                     World(dict(scene="terrain", size=n, spheres=20 * n), seed + 2)]
        st.server = bx.Server(device())
        # which worlds and sizes is the case's own; cameras and worlds are the seed's
        sizes = np.random.default_rng(1000 * n + case["requests"])
        sides = [s for s in (128, 256, 512, 1024) if s <= top]
        st.requests = []
        for _ in range(case["requests"]):
            w = st.worlds[sizes.integers(3)]
            c = scenes.orbit_camera(SimpleNamespace(camera=w.base), r.uniform(), r.uniform())
            cam = bx.camera_perspective(c["position"], c["direction"], c["up"], c["fovy"])
            side = int(sizes.choice(sides))
            st.requests.append((w.world, cam, w.rend, side, side - int(sizes.integers(0, side // 8)),
                                int(sizes.choice([1, 4, 16]))))
        return st
    st.w = World(case, seed)
    if kind in ("frame", "edit"):
        st.frame = bx.Frame(device(), case["w"], case["h"])
        st.channels = [CHANNELS[c] for c in case["read"].split(",")]
        r = np.random.default_rng(seed)
        st.tf = scenes.ramp_tf(256, 0.3 + 0.5 * r.uniform())
    else:
        st.rays = _rays(case, seed)
        st.hits = torch.zeros(case["rays"], 8, device=GPU)
        torch.cuda.synchronize()
    return st


def _trace(st, any_hit):
    bx.check(bx.lib().bnx_trace(st.w.insts.h, st.rays.data_ptr(), len(st.rays), st.hits.data_ptr(),
                                abi.BNX_TRACE_ANY if any_hit else abi.BNX_TRACE_CLOSEST))


def run(st):
    kind = st.case["kind"]
    if kind == "serve":
        tickets = [st.server.submit(*q) for q in st.requests]
        st.server.run_until_idle()
        out = [st.server.read(t, abi.BNX_FB_COLOR_SRGB8) for t in tickets]
        for t in tickets:
            st.server.release(t)
        return out
    if kind in ("frame", "edit"):
        if kind == "edit":
            st.w.vols[0].set_transfer_function(st.tf, (0.0, 1.0), 50.0)
        st.frame.reset()
        bx.render(st.w.world, st.w.cam, st.w.rend, st.frame, st.case["spp"])
        return [st.frame.read(c) for c in st.channels]
    if kind == "build":
        for g in st.w.groups:
            g.build()
        st.w.insts.build()
        _trace(st, False)
        info = [g.info() for g in st.w.groups]
        return {"hit": _hit(st), "depth": [i.max_depth for i in info], "prims": [i.num_prims for i in info]}
    _trace(st, st.case["any"])
    if st.case["any"]:
        # which hit ends an occlusion ray is the traversal's choice: its answer is whether there is one
        device().sync()
        return {"occluded": st.hits.view(torch.int32)[:, 3] >= 0}
    return {"hit": _hit(st)}


def _hit(st):
    return {"t": st.hits[:, 0], "uv": st.hits[:, 1:3], "ids": st.hits.view(torch.int32)[:, 3:8]}


# -------------------------------------------------------------- work, error
def work(case):
    """Bytes: each input record that the rays must meet and each output, once.  Operations: for a ray a descent
    of a 4-wide tree (four slab tests of 18 operations a level), two primitive tests of 50 and a shading step
    of 200; for a ray in a volume 40 collisions of 60 operations (structured), 150 (tets) or 800 (other cells)."""
    n, kind, scene = case["size"], case["kind"], case["scene"]
    if kind == "serve":
        side = 0.5 * case["top"]
        paths = case["requests"] * side * side * 7
        return {"bytes": case["requests"] * side * side * 4.0, "flops": paths * 3 * 900.0}
    prims = {"surface": 20 * 4 ** n + case.get("spheres", 0), "terrain": 2 * (n - 1) ** 2 + case.get("spheres", 0),
             "tubes": 2.5 * n * case.get("copies", 1), "volume": n ** 3, "tets": 5 * n ** 3, "cells": 3 * n ** 3}[scene]
    data = prims * {"surface": 36, "terrain": 36, "tubes": 32, "volume": 4, "tets": 32, "cells": 40}[scene]
    levels = max(1.0, math.log(max(4, prims), 4))
    ray = levels * 72 + 100.0
    if kind in ("trace", "build"):
        rays = case["rays"]
        b = rays * 64 + min(data, rays * 36 * 2.0)
        # a build reads every primitive's record and writes its box, order and share of the nodes
        return {"bytes": b + (prims * (36 + 32 + 4 + 48) if kind == "build" else 0), "flops": rays * ray}
    px = case["w"] * case["h"]
    paths = px * case["spp"]
    size = {"color": 16, "srgb8": 4, "rgba8": 4, "depth": 4, "prim": 4, "inst": 4, "obj": 4, "normal": 12}
    b = px * sum(size[c] for c in case["read"].split(",")) + min(data, paths * 36.0 * 4)
    steps = {"volume": 40 * 60.0, "tets": 40 * 150.0, "cells": 40 * 800.0}.get(scene)
    return {"bytes": b, "flops": paths * 3 * ((steps or ray) + 200)}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """closest hits by brute force in 64 bits, where rays x primitives allow; a rendered frame has no 64-bit value
    (its random walk branches on rounded numbers), nor has an occlusion answer"""
    if case["kind"] != "trace" or case["any"] or case["scene"] != "surface":
        return None
    sc = surface_scene(case, seed)
    m, s = sc.meshes[0], sc.spheres[0]
    if case["rays"] * (len(m.indices) + len(s.radii)) > 4e9:
        return None
    rays = _rays(case, seed).double()
    v = torch.from_numpy(m.vertices).to(GPU).double()[torch.from_numpy(m.indices).long().to(GPU)]
    v0, e1, e2 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    nrm = torch.linalg.cross(e1, e2)
    c, rad = torch.from_numpy(s.centers).to(GPU).double(), torch.from_numpy(s.radii).to(GPU).double()
    out = torch.empty(len(rays), dtype=torch.float64, device=GPU)
    step = max(1, int(2.5e7 // (len(v0) + len(c))))
    for a in range(0, len(rays), step):
        o, d, tm = rays[a:a + step, 0:3], rays[a:a + step, 4:7], rays[a:a + step, 7]
        dn = d @ nrm.T
        t = ((v0 * nrm).sum(1) - o @ nrm.T) / dn
        # barycentrics from triple products of the ray's moment o x d with the edges
        cr = torch.linalg.cross(o, d)
        uu = -(cr @ e2.T + d @ torch.linalg.cross(v0, e2).T) / dn
        vv = (cr @ e1.T + d @ torch.linalg.cross(v0, e1).T) / dn
        ok = (dn != 0) & (t > 0) & (uu >= 0) & (vv >= 0) & (uu + vv < 1)
        best = torch.where(ok, t, torch.inf).amin(1)
        b = (d @ c.T) - (o * d).sum(1, keepdim=True)
        dd = (d * d).sum(1, keepdim=True)
        q = (c * c).sum(1) - 2 * (o @ c.T) + (o * o).sum(1, keepdim=True) - rad * rad
        disc = b * b - dd * q
        root = torch.sqrt(disc.clamp(min=0))
        t1, t2 = (b - root) / dd, (b + root) / dd
        ts = torch.where(t1 > 0, t1, t2)
        ts = torch.where((disc >= 0) & (ts > 0), ts, torch.inf).amin(1)
        out[a:a + step] = torch.minimum(torch.minimum(best, ts), tm)
    return {"hit": {"t": out, "uv": None, "ids": None}}
