"""The batch autotuner tries the plan's own sort (digit width 0: runs merged by rank
for small batches, which no explicit width selects) first, and keeps it unless a width
is faster (host logic, no GPU)."""
import numpy as np
import pytest

from nexusbvh_amd import batch


@pytest.mark.parametrize("ms_by_width,chosen", [
    ({0: 1.0, 8: 1.5, 7: 1.6}, 0),    # a small batch: the merged sort
    ({0: 1.0, 8: 0.99, 7: 1.1}, 0),   # as fast within the tolerance: the default stays
    ({0: 1.0, 8: 1.1, 7: 0.9}, 7),
])
def test_default_sort_is_a_candidate(monkeypatch, ms_by_width, chosen):
    class Plan:
        meshes = 2

        def __init__(self, prims, offsets, config, lanes):
            # other settings make no difference, or a slower one
            self.ms = ms_by_width[config.sortDigitBits] + (0.5 if lanes or config.hplocBlocksPerCu == 8 else 0.0)

        def mesh_sah(self, i):
            return 10.0

        def close(self):
            pass

    monkeypatch.setattr(batch, "BatchPlan", Plan)
    monkeypatch.setattr(batch, "time_plan", lambda plan, reps: plan.ms)
    tuned = batch.autotune(None, np.array([0, 5, 9]))
    assert tuned.config.sortDigitBits == chosen
    assert tuned.trials[0]["digit_bits"] == 0
    assert tuned.ms == ms_by_width[chosen]
