"""GPU tests of the BVH8 either side of 2^20 primitives, where a launch per level takes
over from the expansion of every node: slivers and a surface, 32- and 64-bit keys,
against the oracle, slot for slot.
"""
import pytest

import nxb_checks
from nexusbvh_amd import builder as B
from nexusbvh_amd import native, scenes
from nexusbvh_amd.builder import BuildConfig, DevicePrimitives
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SWITCH = 1 << 20  # the most primitives that are expanded


@pytest.mark.parametrize("n", [SWITCH, SWITCH + 1])
@pytest.mark.parametrize("scene,bits", [("slivers", 64), ("surface", 64), ("surface", 32)])
def test_either_side_of_the_switch(scene, bits, n):
    if native.device_count() == 0:
        pytest.skip("no GPU")
    tris = scenes.slivers(n, seed=91) if scene == "slivers" else scenes.icosphere(n)
    assert len(tris) == n
    bvh = B.BuildBVH8(DevicePrimitives.from_numpy(tris), n, BuildConfig(mortonBits=bits))
    try:
        nodes, prim = B.bvh8_to_host(bvh)
    finally:
        B.FreeDeviceBVH(bvh)
    ref = O.build(tris, 1, bits, 32, 8)
    assert len(nodes) == len(ref["bvh8"])
    assert O.compare_bvh8(nodes, prim, ref["bvh8"], ref["prim_idx"], n)[0] == 0
    nxb_checks.bvh8_invariants(nodes, prim, n)
