"""The march kernels where they can go wrong, on the GPU against the CPU
oracle: frames whose rays do not fill a wave, a 256-ray block or its chunks;
more volumes in a world than a launch has claim counters; scalars that are
not finite (no corner copy, open value ranges); macrocells whose majorants are
as small as floats get; isosurfaces whose samples'
sides come from a fine grid of a single cell up to one a few cells wide, at
values inside, at the ends and outside of the field's range, and over cells
collapsed to triangles and lines, or graded.  IDs, ray and sample counts, depths
and pixels bit for bit; only where ratio tracking passes several volumes, whose
estimates the oracle multiplies volume by volume and the march factor by
factor, pixels within a rounding per factor."""
import dataclasses

import numpy as np
import pytest

import barney_amd as bx
from barney_amd import abi, scenes

pytestmark = pytest.mark.gpu


def _compare(dev, orc, sc, world, scene, spp, flags=0, rtol=0.0):
    rend = abi.renderer(bg=sc.bg_color, ambient=sc.ambient, flags=flags)
    c = sc.camera
    fr = bx.Frame(dev, sc.width, sc.height)
    st = bx.render(world, bx.camera_perspective(c["position"], c["direction"], c["up"], c["fovy"]), rend, fr, spp)
    of = orc.Frame(sc.width, sc.height)
    _, ost = orc.render(scene, orc.camera_perspective(c["position"], c["direction"], c["up"], c["fovy"]), rend, of,
                        spp)
    for ch in (abi.BNX_FB_PRIMID, abi.BNX_FB_INSTID, abi.BNX_FB_OBJID):
        g, r = fr.read(ch), of.read(ch)
        assert np.array_equal(g, r), (ch, int((g != r).sum()))
    assert np.array_equal(fr.read(abi.BNX_FB_DEPTH).view(np.uint32), of.read(abi.BNX_FB_DEPTH).view(np.uint32))
    # accumulated in steps of 2^-32 a sample
    g, r = fr.read(abi.BNX_FB_COLOR), of.read(abi.BNX_FB_COLOR)
    assert np.allclose(g, r, rtol=rtol, atol=2.0 ** -31 if rtol else 0.0), float(np.abs(g - r).max())
    assert st["rays"] == ost["rays"]
    assert st["volume_samples"] == ost["volume_samples"]
    fr.close()


@pytest.mark.parametrize("w,h,flags", [(1, 1, 0), (17, 3, 0), (16, 16, abi.BNX_RENDER_RATIO_TRACKING), (129, 67, 0),
                                       (333, 33, abi.BNX_RENDER_RATIO_TRACKING)])
def test_ray_counts(dev, orc, w, h, flags):
    print(f"march {w}x{h} flags={flags}", flush=True)
    vs = scenes.config2(n=33, mc_grid=8, width=w, height=h)
    _compare(dev, orc, vs, bx.VolumeWorld(dev, vs).world, orc.volume_scene(vs), 1, flags)


@pytest.mark.parametrize("flags", [0, abi.BNX_RENDER_RATIO_TRACKING])
def test_scattered_generations(dev, flags):
    """the later generations of a frame of some millions of rays, which another kernel marches, against the same
    frame in batches below that"""
    print(f"march scattered generations flags={flags}", flush=True)
    w, h, spp = 1000, 900, 9
    vs = scenes.config2(n=33, mc_grid=8, width=w, height=h)
    world, c = bx.VolumeWorld(dev, vs).world, vs.camera
    cam = bx.camera_perspective(c["position"], c["direction"], c["up"], 22.0)
    rend = abi.renderer(bg=vs.bg_color, ambient=vs.ambient, flags=flags)
    tuning, frames, stats = dev.tuning(), [bx.Frame(dev, w, h) for _ in range(3)], []
    try:
        for fr, t in zip(frames, ({}, dict(render_paths=1 << 20, graph_paths=0),
                                  dict(render_paths=1 << 24, graph_paths=1 << 24))):
            dev.set_tuning(**t)
            for _ in range(2):          # the second time a captured loop, if there is one
                fr.reset()
                stats.append(bx.render(world, cam, rend, fr, spp))
    finally:
        dev.set_tuning(**tuning)
    assert stats[0]["rays"] - w * h * spp > 2 << 21
    for st in stats[1:]:
        assert st["rays"] == stats[0]["rays"] and st["volume_samples"] == stats[0]["volume_samples"]
    for ch in (abi.BNX_FB_COLOR, abi.BNX_FB_DEPTH, abi.BNX_FB_OBJID, abi.BNX_FB_NORMAL):
        a, *others = [fr.read(ch) for fr in frames]
        for b in others:
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), ch
    for fr in frames:
        fr.close()


@pytest.mark.parametrize("n,flags", [(2, 0), (11, 0), (11, abi.BNX_RENDER_RATIO_TRACKING)])
def test_many_volumes(dev, orc, n, flags):
    print(f"march of {n} volumes flags={flags}", flush=True)
    vs = scenes.config2(n=17, mc_grid=4, width=40, height=30)
    thin = [dataclasses.replace(vs, grid_origin=(.07 * k, -.05 * k, .03 * k), base_density=vs.base_density / 4)
            for k in range(n)]
    world = bx.World(dev, bx.Group.instances(dev, [], []).build(), vs.dir_lights)
    scene = orc.Scene()
    vols = [bx.Volume(dev, t, user_id=k) for k, t in enumerate(thin)]
    for k, t in enumerate(thin):
        world.add_volume(vols[k], k)
        scene.add_volume(t, user_id=k, user_inst=k)
    scene.set_dir_lights(vs.dir_lights)
    scene.build()
    # up to some hundred factors between 0 and 1, each rounded to 2^-24
    _compare(dev, orc, vs, world, scene, 2, flags, rtol=200 * 2.0 ** -24 if flags else 0.0)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_scalars_not_finite(dev, orc, bad):
    print(f"march scalar {bad}", flush=True)
    vs = scenes.config2(n=20, mc_grid=4, width=48, height=48)
    f = vs.scalars.copy()
    f[9:11, 7, 12] = bad
    vs = dataclasses.replace(vs, scalars=f)
    _compare(dev, orc, vs, bx.VolumeWorld(dev, vs).world, orc.volume_scene(vs), 1)


@pytest.mark.parametrize("flags", [0, abi.BNX_RENDER_RATIO_TRACKING])
@pytest.mark.parametrize("kind", ["structured", "tets"])
def test_tiny_majorants(dev, orc, kind, flags):
    """one narrow Gaussian whose tails run through every exponent down to 0, and a map that begins at 0"""
    print(f"march tiny majorants {kind} flags={flags}", flush=True)
    if kind == "structured":
        vs = scenes.config2(n=64, mc_grid=16, width=64, height=64)
        x = (np.arange(64) / 63.0 - 0.5) ** 2
        r2 = x[:, None, None] + x[None, :, None] + x[None, None, :]
        vs = dataclasses.replace(vs, scalars=np.exp(-r2 / (2 * .05 ** 2)).astype(np.float32))
        world, scene = bx.VolumeWorld(dev, vs).world, orc.volume_scene(vs)
    else:
        vs = scenes.config4(n=16, width=48, height=48)
        r2 = ((vs.vertices.astype(np.float64) - vs.vertices.mean(0)) ** 2).sum(1)
        f = np.exp(-r2 / (2 * (.05 * np.ptp(vs.vertices)) ** 2)).astype(np.float32)
        vs = dataclasses.replace(vs, scalars=f, tf_domain=(0.0, 1.0))
        world, scene = bx.UMeshWorld(dev, vs).world, orc.umesh_scene(vs)
    tails = vs.scalars[(vs.scalars > 0) & (vs.scalars < 1e-38)]
    assert tails.size > 50 and vs.tf[0, 3] == 0
    _compare(dev, orc, vs, world, scene, 2, flags)


@pytest.mark.parametrize("n,iso", [(1, .2), (2, .3), (3, .05), (5, 1.), (5, 0.), (5, -3.), (9, .3)])
@pytest.mark.parametrize("kind", ["tets", "mixed"])
def test_isosurface_sides(dev, orc, kind, n, iso):
    print(f"iso march {kind} n={n} iso={iso}", flush=True)
    make = scenes.config4 if kind == "tets" else scenes.mixed_volume
    us = make(n=n, width=60, height=52, volume=n % 2 == 1)
    lo, hi = float(us.scalars.min()), float(us.scalars.max())
    us = dataclasses.replace(us, iso_value=lo + iso * (hi - lo))      # 0 and 1: the ends of the range
    _compare(dev, orc, us, bx.UMeshWorld(dev, us).world, orc.umesh_scene(us), 1)


@pytest.mark.parametrize("n,mc", [(1, (9, 9, 9)), (6, (5, 40, 17)), (12, (64, 64, 64)), (5, (300, 4, 4)),
                                  (38, (32, 32, 32))])
def test_isosurface_fine_grids(dev, orc, n, mc):
    """few tets with many grid cells each, grids of other shapes than cubes and
    at their largest, tets with more grid cells than they may have ranges in
    (12: some 20,000), and enough tets for a thread each (38)"""
    print(f"iso march fine grid n={n} mc={mc}", flush=True)
    us = dataclasses.replace(scenes.config4(n=n, width=60, height=52, volume=False), mc_dims=mc)
    _compare(dev, orc, us, bx.UMeshWorld(dev, us).world, orc.umesh_scene(us), 1)


@pytest.mark.parametrize("n,power", [(12, 3), (20, 5)])
def test_isosurface_graded_mesh(dev, orc, n, power):
    """cells from far below a fine-grid cell to many of them"""
    print(f"iso march graded mesh n={n} power={power}", flush=True)
    us = scenes.config4(n=n, width=60, height=52, volume=False)
    v = np.round(us.vertices.astype(np.float64) * n) / n                # the lattice without its jitter
    us = dataclasses.replace(us, vertices=(v ** power).astype(np.float32))
    _compare(dev, orc, us, bx.UMeshWorld(dev, us).world, orc.umesh_scene(us), 1)


@pytest.mark.parametrize("n", [4, 8, 14, 40])
def test_isosurface_queries_of_coarse_meshes(dev, n):
    """Tet tests a ray: 46, 34, 27 and 25 when every sub-step up to the crossing
    was queried in turn, each from the last one's tet; the samples that the fine
    grid does not settle have to be far fewer than that, on meshes of few cells
    too (6 to 14)."""
    print(f"iso march queries n={n}", flush=True)
    us = scenes.config4(n=n, width=160, height=120, volume=False)
    world, c, fr = bx.UMeshWorld(dev, us), us.camera, bx.Frame(dev, 160, 120)
    st = bx.render(world.world, bx.camera_perspective(c["position"], c["direction"], c["up"], c["fovy"]),
                   abi.renderer(bg=us.bg_color, ambient=us.ambient), fr, 1)
    fr.close()
    assert st["umesh_tets"] <= 20 * st["rays"], st["umesh_tets"] / st["rays"]


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_isosurface_of_scalars_not_finite(dev, orc, bad):
    print(f"iso march scalar {bad}", flush=True)
    us = scenes.config4(n=6, width=60, height=52)
    f = us.scalars.copy()
    f[len(f) // 2] = bad
    us = dataclasses.replace(us, scalars=f)
    _compare(dev, orc, us, bx.UMeshWorld(dev, us).world, orc.umesh_scene(us), 1)


@pytest.mark.parametrize("kind", ["tets", "mixed"])
@pytest.mark.parametrize("along", [(1,), (1, 7)])
def test_isosurface_of_flat_cells(dev, orc, kind, along):
    """Cells without volume accept points well outside of themselves.  A third
    step along z would fold tets over each other: there a walk's tet and the
    first one of the depth-first query may differ, in any version of the walk,
    so that depths agree with the oracle's only where tets do not overlap."""
    print(f"iso march flat cells {kind} along {along}", flush=True)
    make = scenes.config4 if kind == "tets" else scenes.mixed_volume
    us = make(n=6, width=60, height=52)
    v = us.vertices.copy()
    for k in (57, 114, 171, 200, 235):               # lattice vertices (7 a side) moved onto a neighbour
        for step in along:
            v[k + step] = v[k]
    us = dataclasses.replace(us, vertices=v)
    _compare(dev, orc, us, bx.UMeshWorld(dev, us).world, orc.umesh_scene(us), 1)
