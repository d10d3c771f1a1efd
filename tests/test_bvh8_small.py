"""GPU tests of the BVH8 collapse of small meshes (launches that follow subtrees
inside a block) against the oracle, slot for slot: levels of fewer and of more nodes
than a pass or a block takes, skewed and nested geometry and few first launches; and
of 2^21 primitives and one more, a launch per level.
"""
import numpy as np
import pytest

import nxb_checks
from nexusbvh_amd import builder as B
from nexusbvh_amd import native, scenes
from nexusbvh_amd.builder import BuildConfig, DevicePrimitives
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if native.device_count() == 0:
        pytest.skip("no GPU")


def _check(tris, bits=32, **cfg):
    n = len(tris)
    ref = O.build(tris, 1, bits, 32, 8)
    bvh = B.BuildBVH8(DevicePrimitives.from_numpy(tris), n, BuildConfig(mortonBits=bits, **cfg))
    try:
        nodes, prim = B.bvh8_to_host(bvh)
    finally:
        B.FreeDeviceBVH(bvh)
    assert len(nodes) == len(ref["bvh8"])
    code, where = O.compare_bvh8(nodes, prim, ref["bvh8"], ref["prim_idx"], n)
    assert code == 0, (code, where)
    nxb_checks.bvh8_invariants(nodes, prim, n)
    _check_ranges(nodes, n)


def _check_ranges(nodes, n):
    """primIdx is laid out top-down: a node's leaves at the front of its range,
    then each inner child, in slot order, a range of its primitive count."""
    inner = [[s for s in range(8) if int(nodes["imask"][k]) >> s & 1] for k in range(len(nodes))]
    leaves = [int((nodes["meta"][k] != 0).sum()) - len(inner[k]) for k in range(len(nodes))]
    base = [int(b) for b in nodes["child_base"]]
    count = list(leaves)
    for k in reversed(range(len(nodes))):  # children have larger ids
        for i in range(len(inner[k])):
            assert base[k] + i > k
            count[k] += count[base[k] + i]
    assert count[0] == n
    start = [0] * len(nodes)
    for k in range(len(nodes)):
        if leaves[k]:
            assert int(nodes["prim_base"][k]) == start[k], k
        at = start[k] + leaves[k]
        for i in range(len(inner[k])):
            start[base[k] + i] = at
            at += count[base[k] + i]


@pytest.mark.parametrize("n", [2, 3, 7, 8, 9, 60, 350, 700, 1100, 2003, 5000, 11_000, 30_001])
@pytest.mark.parametrize("scene", ["uniform", "slivers", "blobs"])
def test_small_collapse_sizes(scene, n):
    tris = {"uniform": lambda: scenes.uniform(n, seed=61), "slivers": lambda: scenes.slivers(n, seed=62),
            "blobs": lambda: scenes.blobs_plane(n, seed=63, blobs=5, side=max(1, int((0.15 * n) ** 0.5)), cell=0.3)}[scene]()
    _check(tris, 64 if n % 2 else 32)


def test_small_collapse_nested():
    """Triangles that grow by a constant factor from one point: a long chain of nodes."""
    k = np.arange(700)
    s = (1.09 ** k).astype(np.float32).reshape(-1, 1, 1) * np.float32(1e-12)
    tris = (s * np.array([[1, 0, 0], [0, 1, 0], [0.1, 0.1, 1]], dtype=np.float32)).reshape(-1, 9)
    _check(tris, 64)


def test_small_collapse_duplicates():
    _check(np.repeat(scenes.uniform(60, seed=64), 40, axis=0), 32)


@pytest.mark.parametrize("first", [1, 2, 4])
def test_small_collapse_few_first_launches(monkeypatch, first):
    monkeypatch.setenv("NXB_BVH8_FIRST_LEVELS", str(first))
    _check(scenes.slivers(120_000, seed=65), 32)


@pytest.mark.parametrize("n", [1 << 21, (1 << 21) + 1])
def test_collapse_either_side_of_the_switch(n):
    tris = scenes.uniform(n, seed=66, half_extent=0.002)
    a = B.BuildBVH8(DevicePrimitives.from_numpy(tris), n, BuildConfig(mortonBits=32))
    try:
        nodes, prim = B.bvh8_to_host(a)
    finally:
        B.FreeDeviceBVH(a)
    ref = O.build(tris, 1, 32, 32, 8)
    code, where = O.compare_bvh8(nodes, prim, ref["bvh8"], ref["prim_idx"], n)
    assert code == 0, (code, where)
