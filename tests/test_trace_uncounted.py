"""GPU tests of the traversal without counts (no d_stats): eight lanes per ray and
node up to 2^17 rays, one lane per ray above. Bar as in test_trace.py: the same
triangle and bit-identical t, u and v as the brute force over all triangles.
"""
import numpy as np
import pytest

from nexusbvh_amd import builder as B
from nexusbvh_amd import native, scenes
from nexusbvh_amd.builder import BuildConfig, DevicePrimitives
from nexusbvh_amd.trace import INVALID, TraceClosest, make_rays, random_rays
from oracle import oracle as O

pytestmark = pytest.mark.gpu

GROUP_MAX = 1 << 17  # rays that still take the eight-lane kernel


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if native.device_count() == 0:
        pytest.skip("no GPU")


def _bounds(tris):
    v = tris.reshape(-1, 3)
    return v.min(axis=0), v.max(axis=0)


def _equal(got, ref):
    bad = np.nonzero((got.view(np.uint32).reshape(-1, 4) != ref.view(np.uint32).reshape(-1, 4)).any(axis=1))[0]
    assert bad.size == 0, (int(bad[0]), got[bad[0]], ref[bad[0]])


def _check(tris, rays, cfg=None):
    d = DevicePrimitives.from_numpy(tris)
    bvh = B.BuildBVH8(d, len(tris), cfg or BuildConfig(mortonBits=32))
    try:
        got = TraceClosest(bvh, d, rays)
    finally:
        B.FreeDeviceBVH(bvh)
    ref = O.trace_bruteforce(tris, rays)
    _equal(got, ref)
    return ref


# one ray, around a group block (8 rays), around a wave, either side of the
# switch of kernels (one more leaves a block of one ray), and an odd larger one
@pytest.mark.parametrize("count", [1, 7, 8, 9, 63, 65, 4099, GROUP_MAX, GROUP_MAX + 1, GROUP_MAX + 4099])
def test_uncounted_ray_counts(count):
    tris = scenes.uniform(300, seed=51, half_extent=0.1)
    ref = _check(tris, random_rays(_bounds(tris), count, seed=count))
    assert count < 100 or (ref["prim"] != INVALID).any()


def _both(rays, tris, cfg=None):
    """The rays by themselves and repeated past the switch of kernels."""
    _check(tris, rays, cfg)
    d = DevicePrimitives.from_numpy(tris)
    bvh = B.BuildBVH8(d, len(tris), cfg or BuildConfig(mortonBits=32))
    try:
        few = TraceClosest(bvh, d, rays)
        many = TraceClosest(bvh, d, np.tile(rays, GROUP_MAX // len(rays) + 1))
        counted, _ = TraceClosest(bvh, d, rays, with_stats=True)
    finally:
        B.FreeDeviceBVH(bvh)
    _equal(few, counted)
    _equal(many, np.tile(few, GROUP_MAX // len(rays) + 1))


@pytest.mark.parametrize("scene", ["slivers", "surface", "duplicates", "one", "two"])
def test_uncounted_scenes(scene):
    tris = {"slivers": lambda: scenes.slivers(20_000, seed=52), "surface": lambda: scenes.icosphere(20_000, freq=40),
            # equal distances: the smaller index wins
            "duplicates": lambda: np.repeat(scenes.uniform(700, seed=53, half_extent=0.05), 5, axis=0),
            "one": lambda: scenes.uniform(1, seed=54, half_extent=0.3),
            "two": lambda: scenes.uniform(2, seed=55, half_extent=0.3)}[scene]()
    _both(random_rays(_bounds(tris), 2048, seed=6), tris)


def test_uncounted_axis_rays_and_limits():
    tris = scenes.uniform(4_000, seed=56, half_extent=0.04)
    lo, hi = _bounds(tris)
    rng = np.random.default_rng(7)
    axes = np.concatenate([np.eye(3), -np.eye(3)]).astype(np.float32)
    dirs = axes[rng.integers(0, 6, 2000)]
    dirs[::3] = np.where(dirs[::3] == 0, np.float32(-0.0), dirs[::3])  # negative zeros
    rays = make_rays((lo + rng.random((2000, 3)) * (hi - lo)).astype(np.float32), dirs)
    rays["tmin"] = 0.01
    rays["tmax"] = np.where(rng.random(2000) < 0.5, np.inf, rng.uniform(0.0, 0.3, 2000)).astype(np.float32)
    _both(rays, tris)


def test_uncounted_wide_coordinates():
    """Scene far from the origin and extents over many binades, and rays whose
    direction is not normalised or has tiny components."""
    tris = scenes.uniform(3_000, seed=57, half_extent=0.05)
    tris = (tris.reshape(-1, 3, 3) * np.float32([1000, 1e-3, 30]) + np.float32([5e4, -2, 1e-2])).reshape(-1, 9)
    lo, hi = _bounds(tris)
    rays = random_rays((lo, hi), 2048, seed=8)
    aim = tris[np.random.default_rng(9).integers(0, len(tris), 2048)].reshape(-1, 3, 3).mean(axis=1)
    rays["dir"] = (aim - rays["origin"]) * np.float32(3.0)
    rays["dir"][::5, 1] *= np.float32(1e-25)
    _both(rays, tris)


def test_uncounted_nonfinite_rays_miss():
    tris = scenes.uniform(500, seed=58, half_extent=0.05)
    rays = random_rays(_bounds(tris), 64, seed=10)
    rays["origin"][::4, 0] = np.nan
    rays["dir"][1::4, 2] = np.nan
    rays["dir"][2::4] = 0.0
    rays["tmax"][3::4] = np.nan
    ref = O.trace_bruteforce(tris, rays)
    assert (ref["prim"] == INVALID).all()
    d = DevicePrimitives.from_numpy(tris)
    bvh = B.BuildBVH8(d, len(tris), BuildConfig(mortonBits=32))
    try:
        few = TraceClosest(bvh, d, rays)
        many = TraceClosest(bvh, d, np.tile(rays, GROUP_MAX // 64 + 1))
    finally:
        B.FreeDeviceBVH(bvh)
    assert (few["prim"] == INVALID).all() and (many["prim"] == INVALID).all()


def test_uncounted_child_face_rounded_onto_the_grid():
    from test_trace import _grid_rounding_scene
    tris, rays = _grid_rounding_scene()
    _both(rays, tris)


def test_uncounted_indexed_mesh():
    tris = scenes.icosphere(8_000, freq=25)
    verts, inv = np.unique(tris.reshape(-1, 3), axis=0, return_inverse=True)
    mesh = B.DeviceIndexedMesh.from_numpy(verts.astype(np.float32), inv.reshape(-1, 3).astype(np.uint32))
    rays = random_rays(_bounds(tris), 1500, seed=11)
    bvh = B.BuildBVH8Indexed(mesh, BuildConfig(mortonBits=32))
    try:
        few = TraceClosest(bvh, mesh, rays)
        many = TraceClosest(bvh, mesh, np.tile(rays, 90))
    finally:
        B.FreeDeviceBVH(bvh)
    assert len(many) > GROUP_MAX
    _equal(few, O.trace_bruteforce(tris, rays))
    _equal(many, np.tile(few, 90))
    assert (few["prim"] != INVALID).any()
