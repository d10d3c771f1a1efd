"""GPU test of the BVH8 of a mesh whose nodes lie at very different levels: the limit
of 96 levels is of a node's own level, whatever block of the collapse places it.
"""
import numpy as np
import pytest

import nxb_checks
from nexusbvh_amd import builder as B
from nexusbvh_amd import native
from nexusbvh_amd.builder import BuildConfig, DevicePrimitives
from oracle import oracle as O

MAX_LEVELS = 96  # of a BVH8


def _chain(per_octave, octaves, corner, size):
    """Boxes [corner, corner + s] with s shrinking from `size`: each holds the next."""
    s = (size * 2.0 ** (-np.arange(per_octave * octaves) / per_octave)).reshape(-1, 1)
    return np.concatenate([np.repeat(np.atleast_2d(corner), len(s), 0), corner + s], 1)


def _scatter(rng, count, corner, size):
    p = corner + rng.random((count, 3)) * size * 0.95
    return np.concatenate([p, p + rng.random((count, 3)) * size * 0.05], 1)


def _deep_scene():
    """In the cells of a 4^3 grid: three long chains with 12,001 boxes at their end; a
    short chain around 270 long ones; 200 boxes in each other cell. A block that follows
    one of the three queues many nodes of about level 50 while another queues the 270
    chains' at about 16; those go on for some 50 levels more."""
    rng = np.random.default_rng(1)
    cell = 0.25
    corners = [np.array([i % 4, i // 4 % 4, i // 16]) * cell for i in range(64)]
    spots = 1 + rng.permutation(63)
    out = []
    for i in spots[:3]:
        out += [_chain(24, 16, corners[i], cell * 0.99), _scatter(rng, 12_001, corners[i], cell * 2.0 ** -16 * 0.9)]
    out.append(_chain(16, 2, corners[0], cell * 0.99))
    sub = cell / 4 / 8
    for i in rng.permutation(512)[:270]:
        c = np.array([i % 8, i // 8 % 8, i // 64]) * sub
        out.append(_chain(48, 13, c, sub * 0.99))
        s = sub * 2.0 ** -13 * 0.99 ** np.arange(500).reshape(-1, 1)
        out.append(np.concatenate([np.repeat(c[None], 500, 0), c + s], 1))
    for i in spots[3:]:
        out.append(_scatter(rng, 200, corners[i], cell))
    return np.concatenate(out).astype(np.float32)


def _levels(nodes):
    level = np.zeros(len(nodes), dtype=np.int64)
    inner = np.unpackbits(nodes["imask"][:, None], axis=1).sum(axis=1)
    for k in range(len(nodes)):  # children have larger ids
        first = int(nodes["child_base"][k])
        level[first:first + int(inner[k])] = level[k] + 1
    return int(level.max()) + 1


@pytest.fixture(scope="module")
def scene():
    boxes = _deep_scene()
    return boxes, O.build(boxes, 0, 64, 32, 8)


def test_scene_is_deep_and_within_the_limit(scene):
    assert 70 < _levels(scene[1]["bvh8"]) < MAX_LEVELS - 15


@pytest.mark.gpu
def test_nodes_of_many_levels_side_by_side(scene):
    if native.device_count() == 0:
        pytest.skip("no GPU")
    boxes, ref = scene
    d = DevicePrimitives.from_numpy(boxes)
    for _ in range(5):  # the blocks' order, and so what they share, differs from run to run
        bvh = B.BuildBVH8(d, len(boxes), BuildConfig(mortonBits=64))
        try:
            nodes, prim = B.bvh8_to_host(bvh)
        finally:
            B.FreeDeviceBVH(bvh)
        assert O.compare_bvh8(nodes, prim, ref["bvh8"], ref["prim_idx"], len(boxes))[0] == 0
    nxb_checks.bvh8_invariants(nodes, prim, len(boxes))
