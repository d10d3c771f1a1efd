"""GPU tests of the merged sort (digit_bits 0, small inputs: runs sorted in LDS,
merged by rank) against the oracle's stable sort: whole keys and the whole
permutation are equal. Sizes around a run (2,048), a group of runs (32,768), a
merge block (256) and the ends of its range.
"""
import numpy as np
import pytest

from nexusbvh_amd import native, stages
from oracle import oracle as O

pytestmark = pytest.mark.gpu

RUN, GROUP = 2048, 32768


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if native.device_count() == 0:
        pytest.skip("no GPU")


def _check(keys, begin, end, vals=None):
    bits = keys.dtype.itemsize * 8
    n = len(keys)
    kd = native.DeviceBuffer.from_array(keys)
    vd = native.DeviceBuffer.from_array(vals) if vals is not None else None
    ko, vo = stages.sort_pairs(kd, n, bits, begin, end, 0, values=vd)
    window = (keys >> keys.dtype.type(begin)) & keys.dtype.type((1 << (end - begin)) - 1)
    perm = np.argsort(window, kind="stable").astype(np.uint32)
    assert np.array_equal(ko.to_array(keys.dtype, n), keys[perm])
    assert np.array_equal(vo.to_array(np.uint32, n), perm if vals is None else vals[perm])


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("n", [2, 3, 64, 255, RUN - 1, RUN, RUN + 1, 2 * RUN, 15 * RUN + 257, GROUP - 1, GROUP, GROUP + 1,
                               2 * GROUP + RUN - 1, 3 * GROUP + 17, 5 * 65536, 5 * 65536 + 1, (1 << 19) - 1, 1 << 19,
                               (1 << 19) + 1])
def test_merged_sizes(bits, n):
    """Morton-like windows; the last sizes of each width take the LSD sort."""
    rng = np.random.default_rng(n)
    b, e = O.sort_window(bits)
    _check(rng.integers(0, 2 ** 64, n, dtype=np.uint64).astype(np.uint32 if bits == 32 else np.uint64), b, e)


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("kind", ["equal", "two", "ties", "ascending", "descending", "ones"])
def test_merged_orders(bits, kind):
    """Ties keep their order across runs and groups; keys of all ones beside the fill of a ragged last run."""
    dt = np.uint32 if bits == 32 else np.uint64
    n = 2 * GROUP + 5 * RUN + 77
    rng = np.random.default_rng(3)
    keys = {"equal": np.full(n, 12345), "two": rng.integers(0, 2, n) * 8, "ties": rng.integers(0, 40, n) << 3,
            "ascending": np.arange(n) * 5, "descending": np.arange(n)[::-1] * 5,
            "ones": np.where(rng.random(n) < 0.5, -1, rng.integers(0, 1 << 30, n))}[kind].astype(np.int64).astype(dt)
    b, e = O.sort_window(bits)
    _check(keys, b, e)
    _check(keys, 0, bits)


@pytest.mark.parametrize("begin,end,n", [(0, 64, 100_003), (31, 33, 5_000), (40, 49, 30_001), (20, 60, 70_001), (63, 64, 4_097),
                                         (0, 1, 2_500)])
def test_merged_windows_and_values(begin, end, n):
    """Whole and partial windows, digits across the two words, the caller's values."""
    rng = np.random.default_rng(begin + end)
    keys = rng.integers(0, 2 ** 64, n, dtype=np.uint64)
    _check(keys, begin, end, rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32))
