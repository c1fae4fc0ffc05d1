"""The trace kernels' waves where they can go wrong, against the CPU oracle:
ray counts at the edges of a wave, of a chunk and of a 256-ray block, for
every variant of the ray-array kernel (triangles and spheres, or all
primitives; with and without instance transforms); rays along and against
every axis and rays that are not finite; instances whose transform flattens
them and has no inverse, among others; and rays traced by several threads
of one device at once.  Hits are compared bit for bit."""
import threading

import numpy as np
import pytest

import barney_amd as bx
from barney_amd import abi, scenes
from tests import helpers

pytestmark = pytest.mark.gpu

SPECS = {"plain": helpers.soup_spec, "xf": helpers.instanced_spec,
         "ext": lambda: helpers.sticks_spec(False), "ext_xf": lambda: helpers.sticks_spec(True)}


def _same(g, o):
    bad = helpers.hits_equal(g, o)
    assert len(bad) == 0, (len(bad), g[bad[:3]], o[bad[:3]])


@pytest.mark.parametrize("name", sorted(SPECS))
def test_ray_counts(dev, orc, name):
    spec = SPECS[name]()
    g, o = spec.gpu(dev), spec.oracle(orc)
    rays = scenes.random_rays(21, 8200, radius=6.0, spread=3.0)
    want = o.trace(rays)[0]
    for n in (1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 4095, 4097, 8200):
        print(f"trace waves {name} n={n}", flush=True)
        _same(g.trace(rays[:n]), want[:n])
        hit = g.trace(rays[:n], any_hit=True)
        assert np.array_equal(hit["prim_id"] >= 0, want[:n]["prim_id"] >= 0)


@pytest.mark.parametrize("name,n", [("ext", 100001), ("ext_xf", 180007), ("ext", 700001), ("plain", 100001)])
def test_chunks_of_arrays(dev, orc, name, n):
    """chunks of 32, of 64 and of more rays"""
    print(f"trace waves chunks {name} n={n}", flush=True)
    spec = SPECS[name]()
    rays = scenes.random_rays(25, n, radius=6.0, spread=3.0)
    _same(spec.gpu(dev).trace(rays), spec.oracle(orc).trace(rays)[0])


@pytest.mark.parametrize("name", ["plain", "xf"])
def test_directions(dev, orc, name):
    """all signs of a direction, and components that are 0 or -0"""
    print(f"trace waves directions {name}", flush=True)
    spec = SPECS[name]()
    g, o = spec.gpu(dev), spec.oracle(orc)
    c = np.array([-1.0, -0.0, 0.0, 1.0, 0.3, -0.7], np.float32)
    d = np.array([(x, y, z) for x in c for y in c for z in c if x or y or z], np.float32)
    rays = scenes.random_rays(22, len(d) * 20, radius=6.0, spread=3.0).reshape(len(d), 20, 8)
    rays[:, :, 4:7] = d[:, None, :]
    rays[:, :, 0:3] = np.float32(0.2) * rays[:, :, 0:3] - np.float32(4.0) * d[:, None, :]
    rays = np.ascontiguousarray(rays.reshape(-1, 8))
    want = o.trace(rays)[0]
    assert (want["prim_id"] >= 0).any()
    _same(g.trace(rays), want)


def test_rays_not_finite(dev):
    print("trace waves not finite", flush=True)
    g = helpers.soup_spec().gpu(dev)
    rays = scenes.random_rays(23, 300, radius=5.0, spread=2.0)
    for k, bad in enumerate((np.nan, np.inf, -np.inf)):
        rays[k::3, 0:3] = bad
    assert (g.trace(rays)["prim_id"] == -1).all()
    assert (g.trace(rays, any_hit=True)["prim_id"] == -1).all()


@pytest.mark.parametrize("ext", [False, True])
@pytest.mark.parametrize("flat", [(1, 0, 0, 0, 1, 0, 0, 0, 0), (0, 0, 0, 0, 0, 0, 0, 0, 1), (0,) * 9])
def test_flat_instances(dev, orc, ext, flat):
    """a flattened instance is not hit, and a ray that meets its box goes on
    to the instances behind it: the IDs below and above the flat ones"""
    print(f"trace waves flat instances ext={ext} {flat}", flush=True)
    spec = helpers.sticks_spec(True) if ext else helpers.instanced_spec()
    plain = list(spec.insts)
    m = np.array(list(flat) + [0.1, -0.2, 0.3], np.float32)
    inv = np.full(12, np.nan, np.float32)
    at = (0, 2, len(plain) + 1)
    for k in at:
        spec.insts.insert(k, (plain[-1][0], 90 + k, m, inv))
    rays = scenes.random_rays(24, 20000, radius=6.0, spread=3.0)
    o = spec.oracle(orc)
    want = o.trace(rays)[0]
    hit = want["prim_id"] >= 0
    assert hit.sum() > 1000 and not np.isin(want["inst"], at).any()
    # as without them, but for the places of the others
    spec.insts = plain
    without = spec.oracle(orc).trace(rays)[0]
    assert np.array_equal(want["t"], without["t"]) and np.array_equal(want["prim_id"], without["prim_id"])
    for k in at:
        spec.insts = spec.insts[:k] + [(plain[-1][0], 90 + k, m, inv)] + spec.insts[k:]
    g = spec.gpu(dev)
    _same(g.trace(rays), want)
    assert np.array_equal(g.trace(rays, any_hit=True)["prim_id"] >= 0, hit)


@pytest.mark.parametrize("kind", ["plain", "cylinders", "volume"])
def test_many_rays_few_primitives(dev, kind):
    """a batch that keeps one ray per thread against the same frame in batches too small for that"""
    print(f"trace waves few primitives {kind}", flush=True)
    w, h = 653, 461
    sc = scenes.config1(width=w, height=h, subdiv=3)   # 2,280 primitives
    if kind == "cylinders":
        sc.cylinders.append(scenes.sticks(300))
    world, c = bx.SurfaceWorld(dev, sc), sc.camera
    if kind == "volume":
        vs = scenes.config2(n=17, mc_grid=4, width=w, height=h)
        vol = bx.Volume(dev, vs)
        world.world.add_volume(vol, 3)
    cam = bx.camera_perspective(c["position"], c["direction"], c["up"], c["fovy"])
    rend = abi.renderer(bg=sc.bg_color, ambient=sc.ambient)
    tuning, frames, stats = dev.tuning(), [bx.Frame(dev, w, h) for _ in range(3)], []
    assert w * h < 1 << 19 <= 2 * w * h
    try:
        for fr, t in zip(frames, ({}, dict(graph_paths=0), dict(render_paths=1 << 18))):
            dev.set_tuning(**t)
            stats.append(bx.render(world.world, cam, rend, fr, 2))
    finally:
        dev.set_tuning(**tuning)
    assert len({st["rays"] for st in stats}) == 1
    for ch in (abi.BNX_FB_COLOR, abi.BNX_FB_DEPTH, abi.BNX_FB_PRIMID, abi.BNX_FB_INSTID, abi.BNX_FB_NORMAL):
        a, *others = [fr.read(ch) for fr in frames]
        for b in others:
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), ch
    for fr in frames:
        fr.close()


def test_threads(dev, orc):
    print("trace waves threads", flush=True)
    spec = helpers.soup_spec()
    g, o = spec.gpu(dev), spec.oracle(orc)
    sets = [scenes.random_rays(30 + k, 30000 + 777 * k, radius=5.0, spread=2.0) for k in range(4)]
    want = [o.trace(r)[0] for r in sets]
    got = [[] for _ in sets]

    def work(k):
        for _ in range(4):
            got[k].append(g.trace(sets[k]))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(sets))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, w in enumerate(want):
        assert len(got[k]) == 4
        for h in got[k]:
            _same(h, w)
