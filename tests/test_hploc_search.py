"""GPU tests of H-PLOC's neighbour search and node stores against the oracle,
byte for byte: areas that overflow to infinity or are NaN (the search then masks
its candidates explicitly) alone and among finite ones, every kind of radius,
short groups, and either side of the switch to staged wide records.
"""
import numpy as np
import pytest

from nexusbvh_amd import builder as B
from nexusbvh_amd import native, scenes, stages
from nexusbvh_amd.builder import BuildConfig, DevicePrimitives, MergeMode
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if native.device_count() == 0:
        pytest.skip("no GPU")


def _boxes(n, kind, seed):
    """Leaf boxes: all huge (areas overflow), huge and flat (infinite times
    zero), or small ones with every 97th or every second huge."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-1, 1, (n, 3))
    e = rng.uniform(0.001, 0.01, (n, 3))
    if kind == "flat":
        e[:, 2] = 0
        c[:, 2] = 0
    scale = np.ones(n)
    scale[:: {"huge": 1, "flat": 1, "rare": 97, "half": 2}[kind]] = 3e38
    lo, hi = (c - e) * scale[:, None], (c + e) * scale[:, None]
    return np.hstack([np.clip(lo, -3e38, 3e38), np.clip(hi, -3e38, 3e38)]).astype(np.float32)


@pytest.mark.parametrize("mode", [MergeMode.WAVE32, MergeMode.WAVE64])
@pytest.mark.parametrize("radius", [1, 3, 8, 16, "table"])
@pytest.mark.parametrize("kind,n", [("huge", 3001), ("flat", 700), ("rare", 20_011), ("half", 5000)])
def test_search_with_areas_that_overflow(kind, n, radius, mode):
    width = 32 if mode == MergeMode.WAVE32 else 64
    boxes = _boxes(n, kind, n)
    nodes0, _, bad = O.scene_bounds(boxes, 0)
    assert not bad
    rng = np.random.default_rng(7)
    keys = np.sort(rng.integers(0, 1 << 63, n, dtype=np.uint64))
    perm = rng.permutation(n).astype(np.uint32)
    cfg, kw, r = BuildConfig(mergeMode=mode), {}, 8
    if radius == "table":
        table = rng.choice(np.array([0, 1, 2, 4, 8, 16], dtype=np.uint8), (n >> 8) + 1)
        tbl = native.DeviceBuffer.from_array(table)
        cfg = BuildConfig(mergeMode=mode, radiusPolicy=B.RadiusPolicy.TABLE, radiusTable=tbl, radiusTableLen=len(table),
                          segmentLog2=8)
        kw = dict(table=table, seg_log2=8)
    else:
        cfg, r = BuildConfig(mergeMode=mode, searchRadius=radius), radius
    ref = O.hploc(keys, perm, nodes0, width, r, **kw)
    nodes = native.DeviceBuffer.from_array(np.concatenate([nodes0[:n], nodes0[: n - 1]]))
    print("overflow", kind, n, radius, mode.name, flush=True)
    stages.hploc(native.DeviceBuffer.from_array(keys), native.DeviceBuffer.from_array(perm), n, 64, nodes, cfg)
    assert stages.nodes_to_host(nodes, 2 * n - 1).tobytes() == ref[: 2 * n - 1].tobytes()


@pytest.mark.parametrize("n", [2, 3, 17, 33, 34, 65, 130, 1025])
@pytest.mark.parametrize("mode", [MergeMode.WAVE32, MergeMode.WAVE64])
def test_short_groups(n, mode):
    tris = scenes.uniform(n, seed=n)
    ref = O.build(tris, 1, 64, 32 if mode == MergeMode.WAVE32 else 64, 8)
    bvh = B.BuildBVH2(DevicePrimitives.from_numpy(tris), n, BuildConfig(mortonBits=64, mergeMode=mode))
    h = B.ToHost(bvh)
    B.FreeDeviceBVH(bvh)
    assert h.nodes.tobytes() == ref["nodes"][: 2 * n - 1].tobytes()
    B.FreeHostBVH(h)


@pytest.mark.parametrize("n,mode", [(3 * 2 ** 20 - 1, MergeMode.WAVE64), (3 * 2 ** 20, MergeMode.WAVE64),
                                    (3 * 2 ** 20 + 1, MergeMode.WAVE32)])
def test_either_side_of_staged_records(n, mode):
    tris = scenes.uniform(n, seed=67, half_extent=0.002)
    print("staged records", n, mode.name, flush=True)
    bvh = B.BuildBVH8(DevicePrimitives.from_numpy(tris), n, BuildConfig(mortonBits=32, mergeMode=mode))
    try:
        nodes, prim = B.bvh8_to_host(bvh)
    finally:
        B.FreeDeviceBVH(bvh)
    ref = O.build(tris, 1, 32, 32 if mode == MergeMode.WAVE32 else 64, 8)
    assert O.compare_bvh8(nodes, prim, ref["bvh8"], ref["prim_idx"], n)[0] == 0


@pytest.mark.parametrize("mode", [MergeMode.WAVE32, MergeMode.WAVE64])
@pytest.mark.parametrize("above", [1, 8, 16])
@pytest.mark.parametrize("radii,seg_log2", [([8], 6), ([16], 5), ([4, 8], 4), ([2, 8, 16], 6), ([0, 1, 16], 8)])
def test_radius_tables(radii, seg_log2, above, mode):
    """Tables that give a wave's two tasks the same radius or different ones."""
    n = 9_001
    keys = np.sort(np.random.default_rng(8).integers(0, 1 << 63, n, dtype=np.uint64))
    nodes0, _, _ = O.scene_bounds(scenes.uniform(n, seed=85), 1)
    perm = np.random.default_rng(9).permutation(n).astype(np.uint32)
    table = np.random.default_rng(10).choice(np.array(radii, dtype=np.uint8), (n >> seg_log2) + 1)
    tbl = native.DeviceBuffer.from_array(table)
    cfg = BuildConfig(mergeMode=mode, searchRadius=above, radiusPolicy=B.RadiusPolicy.TABLE, radiusTable=tbl,
                      radiusTableLen=len(table), segmentLog2=seg_log2)
    ref = O.hploc(keys, perm, nodes0, 32 if mode == MergeMode.WAVE32 else 64, above, table=table, seg_log2=seg_log2)
    nodes = native.DeviceBuffer.from_array(np.concatenate([nodes0[:n], nodes0[: n - 1]]))
    stages.hploc(native.DeviceBuffer.from_array(keys), native.DeviceBuffer.from_array(perm), n, 64, nodes, cfg)
    assert stages.nodes_to_host(nodes, 2 * n - 1).tobytes() == ref[: 2 * n - 1].tobytes()
