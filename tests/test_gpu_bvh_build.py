"""GPU BVH builder against the CPU specification where its two phases meet:
sizes around the block-built task size (1024) and its multiples, boxes in an
order that puts whole waves into one bin, clusters that split off a few
primitives at a time, equal centroids (median splits through both phases),
every leaf size the entry point takes, and the scratch that stays.  Trees are compared node for node,
orders slot for slot."""
import numpy as np
import pytest
import torch

import barney_amd as bx
from tests import helpers

pytestmark = pytest.mark.gpu


def _boxes(kind, n, seed):
    r = np.random.default_rng(seed)
    if kind == "random":
        return helpers.random_boxes(seed, n)
    if kind == "rows":                      # a mesh's order: runs of slots share two of the three bins
        i = np.arange(n)
        c = np.stack([i % 211, (i // 211) % 7, i // (211 * 7)], 1).astype(np.float32)
    elif kind == "clusters":                # distances over many powers of two: planes that peel the far ones off
        c = (2.0 ** r.uniform(-20, 6, (n, 1)) * r.normal(size=(n, 3))).astype(np.float32)
    else:                                   # "same": no valid plane anywhere
        c = np.full((n, 3), 3.25, np.float32)
    e = r.uniform(0.01, 0.6, (n, 3)).astype(np.float32)
    return np.concatenate([c - e, c + e], 1).astype(np.float32) if kind != "same" else \
        np.concatenate([c - 0.5, c + 0.5], 1).astype(np.float32)


@pytest.mark.parametrize("kind,n,leaf", [
    ("random", 2, 1), ("random", 63, 7), ("random", 64, 1), ("random", 65, 2), ("random", 1023, 4),
    ("random", 1024, 1), ("random", 1025, 1), ("random", 2047, 4), ("random", 2048, 4), ("random", 2049, 4),
    ("random", 30011, 3), ("rows", 5000, 4), ("rows", 40000, 4), ("clusters", 1500, 1), ("clusters", 20000, 4),
    ("same", 1025, 4), ("same", 5003, 1)])
def test_builder_phases(dev, orc, kind, n, leaf):
    print(f"builder {kind} n={n} leaf={leaf}", flush=True)
    boxes = _boxes(kind, n, n + leaf)
    gn, go, ginfo = bx.bvh_build_boxes(dev, boxes, leaf)
    on, oo, od = orc.bvh_build_boxes(boxes, leaf)
    assert np.array_equal(go, oo)
    assert helpers.canonical_bvh(gn, go, leaf) == helpers.canonical_bvh(on, oo, leaf)
    assert ginfo.max_depth == od and ginfo.num_nodes == len(on)


def test_large_builds_give_their_scratch_back(dev):
    """20M boxes need some 1.6 GB of scratch; of that no more than 1 GiB may stay"""
    print("builder scratch of 20M boxes", flush=True)
    bx.bvh_build_boxes(dev, _boxes("random", 5000, 1), 4)
    before = torch.cuda.mem_get_info(0)[0]
    r = np.random.default_rng(5)
    c = r.random((20 << 20, 3), np.float32)
    _, _, info = bx.bvh_build_boxes(dev, np.concatenate([c, c + np.float32(.001)], 1), 4)
    assert info.num_nodes > 5 << 20
    assert before - torch.cuda.mem_get_info(0)[0] < (1024 + 64) << 20
    # and the next build has its scratch again
    boxes = _boxes("random", 3000, 2)
    a, b = bx.bvh_build_boxes(dev, boxes, 4), bx.bvh_build_boxes(dev, boxes, 4)
    assert np.array_equal(a[1], b[1]) and helpers.canonical_bvh(a[0], a[1], 4) == helpers.canonical_bvh(b[0], b[1], 4)
