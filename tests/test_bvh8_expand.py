"""GPU tests of the BVH8 of small meshes made from every node's expansion, against
the oracle, slot for slot: a pass's 32 nodes and a block's 256 queued ones, long
chains, both slot assignments, few first launches, and either side of the switch
to collapsing a level at a time (2^20 primitives).
"""
import numpy as np
import pytest

import nxb_checks
from nexusbvh_amd import builder as B
from nexusbvh_amd import native, scenes
from nexusbvh_amd.builder import BuildConfig, DevicePrimitives, SlotAssignment
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SWITCH = 1 << 20


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if native.device_count() == 0:
        pytest.skip("no GPU")


def _build(tris, **cfg):
    bvh = B.BuildBVH8(DevicePrimitives.from_numpy(tris), len(tris), BuildConfig(mortonBits=32, **cfg))
    try:
        return B.bvh8_to_host(bvh)
    finally:
        B.FreeDeviceBVH(bvh)


def _check(tris, **cfg):
    nodes, prim = _build(tris, **cfg)
    ref = O.build(tris, 1, 32, 32, 8)
    assert len(nodes) == len(ref["bvh8"])
    code, where = O.compare_bvh8(nodes, prim, ref["bvh8"], ref["prim_idx"], len(tris))
    assert code == 0, (code, where)
    nxb_checks.bvh8_invariants(nodes, prim, len(tris))


@pytest.mark.parametrize("n", [2, 4, 9, 33, 150, 260, 1200, 2500, 9000, 65_537, 262_145])
def test_expanded_sizes(n):
    _check(scenes.uniform(n, seed=n))


def test_expanded_chain():
    s = (1.05 ** np.arange(1500)).astype(np.float32).reshape(-1, 1, 1) * np.float32(1e-18)
    _check((s * np.array([[1, 0, 0], [0, 1, 0], [0.1, 0.1, 1]], dtype=np.float32)).reshape(-1, 9))


@pytest.mark.parametrize("first", [1, 3])
def test_expanded_few_first_launches(monkeypatch, first):
    monkeypatch.setenv("NXB_BVH8_FIRST_LEVELS", str(first))
    _check(scenes.slivers(90_000, seed=81))


@pytest.mark.parametrize("slots", [SlotAssignment.GREEDY, SlotAssignment.AUCTION])
def test_expanded_equals_repeated(slots):
    """The same nodes every time, up to their numbering: sorted node bounds and
    exponents, slot masks and metas do not depend on the launches' order."""
    tris = scenes.slivers(50_000, seed=82)
    runs = [_build(tris, slotAssignment=slots) for _ in range(2)]
    key = [np.sort(r[0].view(np.uint8).reshape(len(r[0]), 80)[:, np.r_[0:16, 24:80]].copy().view("V72").ravel())
           for r in runs]
    assert (key[0] == key[1]).all()
    for nodes, prim in runs:
        nxb_checks.bvh8_invariants(nodes, prim, len(tris))


@pytest.mark.parametrize("n", [SWITCH, SWITCH + 1])
def test_either_side_of_expansion(n):
    tris = scenes.uniform(n, seed=83, half_extent=0.002)
    nodes, prim = _build(tris)
    ref = O.build(tris, 1, 32, 32, 8)
    assert O.compare_bvh8(nodes, prim, ref["bvh8"], ref["prim_idx"], n)[0] == 0


def test_levels_with_auction_slots():
    n = SWITCH + 777
    tris = scenes.slivers(n, seed=84)
    nodes, prim = _build(tris, slotAssignment=SlotAssignment.AUCTION)
    a8, ap = O.collapse_bvh8(O.build(tris, 1, 32, 32, 8)["nodes"], n, 1)
    assert O.compare_bvh8(nodes, prim, a8, ap, n)[0] == 0
