"""GPU tests of a batch's BVH8 levels against the oracle, mesh by mesh and slot for
slot: a level of less than a wave, of parts of a block and of several blocks, blocks
whose nodes belong to many trees, and a chain that goes on when all others have ended.
"""
import numpy as np
import pytest

from nexusbvh_amd import batch, native, scenes
from nexusbvh_amd.builder import BuildConfig, DevicePrimitives, SlotAssignment
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if native.device_count() == 0:
        pytest.skip("no GPU")


def _chain(n):
    s = (1.05 ** np.arange(n)).astype(np.float32).reshape(-1, 1, 1) * np.float32(1e-18)
    return (s * np.array([[1, 0, 0], [0, 1, 0], [0.1, 0.1, 1]], dtype=np.float32)).reshape(-1, 9)


@pytest.mark.parametrize("slots", [SlotAssignment.GREEDY, SlotAssignment.AUCTION])
@pytest.mark.parametrize("sizes", [
    [2],
    [70, 2, 9],
    [300] * 5 + [2] * 300,                    # the second level: five trees, then nothing
    [8, 9, 64, 65, 66, 257, 2000, 1025] * 9,  # blocks of 256 nodes across trees
    [-700, 40, 3000, -90, 2, 20_000],         # negative: a chain of that many triangles
])
def test_levels_of_mixed_trees(sizes, slots):
    tris = [_chain(-n) if n < 0 else scenes.slivers(n, seed=500 + i) for i, n in enumerate(sizes)]
    offsets = np.concatenate([[0], np.cumsum([len(t) for t in tris])]).astype(np.uint32)
    plan = batch.BatchPlan(DevicePrimitives.from_numpy(np.concatenate(tris)), offsets,
                           BuildConfig(mortonBits=32, slotAssignment=slots))
    plan.run()
    for m, t in enumerate(tris):
        nodes, prim = plan.mesh_to_host(m)
        ref = O.build(t, 1, 32, 32, 8)
        if slots == SlotAssignment.AUCTION:
            ref["bvh8"], ref["prim_idx"] = O.collapse_bvh8(ref["nodes"], len(t), 1)
        code, where = O.compare_bvh8(nodes, prim, ref["bvh8"], ref["prim_idx"], len(t))
        assert code == 0, (m, len(t), code, where)
