"""GPU tests of the traversal without counts where distances along an axis overflow:
coordinates from 3e8 to 1e12 with zero direction components (whose reciprocal stands
in as 1e30), and tiny directions. Every kernel of it (four, two and one nodes a step,
one lane per ray) and the counted one give the triangle, t, u and v of the brute
force, bit for bit.
"""
import numpy as np
import pytest

from nexusbvh_amd import builder as B
from nexusbvh_amd import native, scenes
from nexusbvh_amd.builder import BuildConfig, DevicePrimitives
from nexusbvh_amd.trace import INVALID, TraceClosest, make_rays
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# rays above which the next kernel takes over: four, two, one node a step, one lane
SWITCHES = (1 << 13, 1 << 15, 1 << 17)


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if native.device_count() == 0:
        pytest.skip("no GPU")


def _check_all_kernels(tris, rays):
    ref = O.trace_bruteforce(tris, rays)
    assert (ref["prim"] != INVALID).sum() >= 20
    d = DevicePrimitives.from_numpy(tris)
    bvh = B.BuildBVH8(d, len(tris), BuildConfig(mortonBits=32))
    try:
        results = {"counted": TraceClosest(bvh, d, rays, with_stats=True)[0], "few": TraceClosest(bvh, d, rays)}
        for above in SWITCHES:
            reps = above // len(rays) + 1
            results[f"above {above}"] = TraceClosest(bvh, d, np.tile(rays, reps))
    finally:
        B.FreeDeviceBVH(bvh)
    for name, got in results.items():
        want = np.tile(ref, len(got) // len(ref))
        bad = np.nonzero((got.view(np.uint32).reshape(-1, 4) != want.view(np.uint32).reshape(-1, 4)).any(axis=1))[0]
        assert bad.size == 0, (name, bad.size, int(bad[0]), got[bad[0]], want[bad[0]])


@pytest.mark.parametrize("size", [3e8, 5e8, 1e9, 1e10, 1e12])
def test_zero_components_of_large_scenes(size):
    tris = (scenes.uniform(300, seed=71, half_extent=0.15) * np.float32(size)).astype(np.float32)
    lo, hi = tris.reshape(-1, 3).min(axis=0), tris.reshape(-1, 3).max(axis=0)
    rng = np.random.default_rng(72)
    axes = np.concatenate([np.eye(3), -np.eye(3)]).astype(np.float32)
    dirs = axes[rng.integers(0, 6, 600)]
    dirs[200:400] = np.where(dirs[200:400] == 0, np.float32(-0.0), dirs[200:400])  # negative zeros
    dirs[400:] += axes[rng.integers(0, 6, 200)]  # one or two components in use
    rays = make_rays((lo + rng.random((600, 3)) * (hi - lo)).astype(np.float32), dirs)
    _check_all_kernels(tris, rays)


# all three axes overflow at once, and the hits' distances do not (components stay
# above 1e-30, below which they count as that)
@pytest.mark.parametrize("size,length", [(3e11, 3e-28), (1e12, 1e-27)])
def test_tiny_directions_in_large_scenes(size, length):
    tris = (scenes.uniform(300, seed=73, half_extent=0.15) * np.float32(size)).astype(np.float32)
    lo, hi = tris.reshape(-1, 3).min(axis=0), tris.reshape(-1, 3).max(axis=0)
    rng = np.random.default_rng(74)
    dirs = rng.normal(size=(600, 3))
    dirs += np.copysign(0.05, dirs)
    dirs *= length / np.linalg.norm(dirs, axis=1, keepdims=True)
    rays = make_rays((lo + rng.random((600, 3)) * (hi - lo)).astype(np.float32), dirs.astype(np.float32), tmax=3e38)
    _check_all_kernels(tris, rays)
