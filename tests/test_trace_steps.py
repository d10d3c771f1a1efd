"""GPU tests of the traversals that take four (up to 2^13 rays), two (up to 2^15)
and one node of a ray a step: the same rays through each give the hits of the
counted traversal bit for bit, on soups and indexed meshes, deep trees and the
ray counts either side of the switches.
"""
import numpy as np
import pytest

from nexusbvh_amd import builder as B
from nexusbvh_amd import native, scenes
from nexusbvh_amd.builder import BuildConfig, DeviceIndexedMesh, DevicePrimitives
from nexusbvh_amd.trace import INVALID, TraceClosest, random_rays

pytestmark = pytest.mark.gpu

QUAD, PAIR = 1 << 13, 1 << 15


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if native.device_count() == 0:
        pytest.skip("no GPU")


def _nested(n):
    """Triangles that grow by a constant factor from one point: a deep tree."""
    s = (1.09 ** np.arange(n)).astype(np.float32).reshape(-1, 1, 1) * np.float32(1e-12)
    return (s * np.array([[1, 0, 0], [0, 1, 0], [0.1, 0.1, 1]], dtype=np.float32)).reshape(-1, 9)


SCENES = {"uniform": lambda: scenes.uniform(30_000, seed=71, half_extent=0.03),
          "slivers": lambda: scenes.slivers(20_000, seed=72),
          "duplicates": lambda: np.repeat(scenes.uniform(900, seed=73, half_extent=0.05), 4, axis=0),
          "nested": lambda: _nested(700)}


def _bits(hits):
    return hits.view(np.uint32).reshape(-1, 4)


@pytest.mark.parametrize("scene", sorted(SCENES))
def test_node_counts_per_step_agree(scene):
    tris = SCENES[scene]()
    v = tris.reshape(-1, 3)
    rays = random_rays((v.min(axis=0), v.max(axis=0)), 1500, seed=9)
    if scene == "nested":  # across the chain, at every scale
        k = np.arange(1500) % 700
        c = tris.reshape(-1, 3, 3).mean(axis=1)[k]
        rays["origin"] = c * np.float32(1.7)
        rays["dir"] = -c / np.linalg.norm(c, axis=1, keepdims=True)
    d = DevicePrimitives.from_numpy(tris)
    bvh = B.BuildBVH8(d, len(tris), BuildConfig(mortonBits=64))
    try:
        ref, _ = TraceClosest(bvh, d, rays, with_stats=True)
        for count in (1, 2, 3, 1500, QUAD, QUAD + 1, PAIR, PAIR + 1):
            many = np.resize(rays, count)
            got = TraceClosest(bvh, d, many)
            assert np.array_equal(_bits(got), np.resize(_bits(ref), (count, 4))), count
    finally:
        B.FreeDeviceBVH(bvh)
    assert (ref["prim"] != INVALID).any()


@pytest.mark.parametrize("count", [5, QUAD + 3, PAIR + 5])
def test_indexed_mesh_agrees(count):
    tris = scenes.icosphere(20_000, freq=40)
    v, i = np.unique(tris.reshape(-1, 3), axis=0, return_inverse=True)
    mesh = DeviceIndexedMesh.from_numpy(v.astype(np.float32), i.reshape(-1, 3).astype(np.uint32))
    rays = np.resize(random_rays((v.min(axis=0), v.max(axis=0)), 2000, seed=10), count)
    bvh = B.BuildBVH8Indexed(mesh, BuildConfig(mortonBits=32))
    try:
        ref, _ = TraceClosest(bvh, mesh, rays, with_stats=True)
        got = TraceClosest(bvh, mesh, rays)
    finally:
        B.FreeDeviceBVH(bvh)
    assert np.array_equal(_bits(got), _bits(ref))
