"""Unstructured volumes with pyramids, prisms and hexahedra besides tets
(UMeshField::DD::eltScalar, umesh/common/UMeshField.h:372-495, with the
Newton inversions of ElementIntersection.h) on the GPU against the CPU
oracle: macrocell value ranges and majorants bit-exact (tets rasterized
split, other cells by their boxes), then 1-spp frames of the volume and an
isosurface over it -- primary IDs bit-exact, depth within 1e-5 relative,
pixels within 1e-3, and the same rays and volume samples -- on a jittered
mesh (non-planar faces: neighbouring cells overlap or leave gaps, where the
first cell of the depth-first query decides) and on a planar-faced one."""
import dataclasses

import numpy as np
import pytest

import barney_amd as bx
from barney_amd import abi, scenes

pytestmark = pytest.mark.gpu

MESHES = {
    "jittered": dict(n=8, jitter=0.15),
    "planar": dict(n=7, jitter=0.0),
    "hex_pyr": dict(n=6, jitter=0.1, kinds=(scenes.CELL_HEX, scenes.CELL_PYR)),
}


def _scene(name, w=96, h=96, volume=True):
    return scenes.mixed_volume(width=w, height=h, volume=volume, **MESHES[name])


@pytest.mark.parametrize("name", sorted(MESHES))
def test_cell_macrocells_match(dev, orc, name):
    print(f"mixed cells macrocells {name}", flush=True)
    us = _scene(name)
    g = bx.Volume(dev, us)
    gd, glo, ghi = g.mc_ranges()
    o = orc.umesh_scene(us)
    od, olo, ohi = o.mc_ranges(0)
    assert tuple(gd) == tuple(od)
    assert np.array_equal(glo.view(np.uint32), olo.view(np.uint32))
    assert np.array_equal(ghi.view(np.uint32), ohi.view(np.uint32))
    _, gm = g.majorants()
    _, om = o.volume_majorants(0)
    assert np.array_equal(gm.view(np.uint32), om.view(np.uint32))


@pytest.mark.parametrize("name,volume", [("jittered", True), ("jittered", False), ("planar", True),
                                         ("hex_pyr", True)])
def test_cell_one_spp_parity(dev, orc, name, volume):
    print(f"mixed cells 1spp {name} volume={volume}", flush=True)
    us = _scene(name, volume=volume)
    rend = abi.renderer(bg=us.bg_color, ambient=us.ambient)
    w = bx.UMeshWorld(dev, us)
    cam = bx.camera_perspective(us.camera["position"], us.camera["direction"], us.camera["up"], us.camera["fovy"])
    fr = bx.Frame(dev, us.width, us.height)
    st = bx.render(w.world, cam, rend, fr, 1)
    o = orc.umesh_scene(us)
    ocam = orc.camera_perspective(us.camera["position"], us.camera["direction"], us.camera["up"], us.camera["fovy"])
    of = orc.Frame(us.width, us.height)
    _, ost = orc.render(o, ocam, rend, of, 1)
    for ch in (abi.BNX_FB_PRIMID, abi.BNX_FB_INSTID, abi.BNX_FB_OBJID):
        g, r = fr.read(ch), of.read(ch)
        assert np.array_equal(g, r), (ch, int((g != r).sum()))
    obj = of.read(abi.BNX_FB_OBJID)
    assert (obj == us.iso_user_id).sum() > 50
    if volume:
        assert (obj == us.user_id).sum() > 50
    assert np.allclose(fr.read(abi.BNX_FB_DEPTH), of.read(abi.BNX_FB_DEPTH), rtol=1e-5, atol=0)
    d = np.abs(fr.read(abi.BNX_FB_COLOR) - of.read(abi.BNX_FB_COLOR))
    print("mixed cells 1spp max abs diff", float(d.max()), flush=True)
    assert d.max() <= 1e-3
    assert st["rays"] == ost["rays"]
    assert st["volume_samples"] == ost["volume_samples"]
    fr.close()


def test_cells_of_huge_determinants(dev, orc):
    """cells some 2^42 across, whose Jacobian's determinants have no normal reciprocal"""
    print("mixed cells 1spp of huge cells", flush=True)
    us = scenes.mixed_volume(n=4, width=48, height=48, jitter=0.05, kinds=(scenes.CELL_HEX,))
    scale = np.float32(4 * 5.0e12)
    cells = (us.vertices * scale).astype(np.float32)
    c = {k: tuple(float(x) * float(scale) for x in v) if k in ("position", "direction", "target") else v
         for k, v in us.camera.items()}
    us = dataclasses.replace(us, vertices=cells, base_density=us.base_density / float(scale), camera=c)
    rend = abi.renderer(bg=us.bg_color, ambient=us.ambient)
    frames = []
    for side, o, scene in ((bx, dev, bx.UMeshWorld(dev, us)), (orc, None, orc.umesh_scene(us))):
        cam = side.camera_perspective(c["position"], c["direction"], c["up"], c["fovy"])
        fr = bx.Frame(dev, 48, 48) if o else orc.Frame(48, 48)
        st = bx.render(scene.world, cam, rend, fr, 1) if o else orc.render(scene, cam, rend, fr, 1)[1]
        frames.append((st["rays"], st["volume_samples"], fr.read(abi.BNX_FB_OBJID), fr.read(abi.BNX_FB_COLOR)))
    g, r = frames
    assert (r[2] == us.iso_user_id).sum() > 30 and (r[2] == us.user_id).sum() > 1000
    assert g[0] == r[0] and g[1] == r[1] and np.array_equal(g[2], r[2])
    assert np.abs(g[3] - r[3]).max() <= 1e-3
