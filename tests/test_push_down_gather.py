"""Multimap directory scan at tile and look-back edges; push-down probes that
gather their rows first, at trip edges, thresholds and split list lengths."""
import pytest

from dogqc_amd import runtime as rt
from tests.test_gpu_parity import check, workloadAcc

pytestmark = pytest.mark.gpu


# 4096 buckets a tile; 64 tiles a look-back step
@pytest.mark.parametrize("buckets", [1, 63, 4095, 4096, 4097, 64 * 4096, 64 * 4096 + 1, 200 * 4096 + 17])
@pytest.mark.parametrize("plan", ["c2_none", "c2_pushdown"])
def test_directory_scan(buckets, plan):
    acc = workloadAcc("c2", {"build": 3000, "probe": 5000}, seed=buckets)
    t = rt.newTuning()
    t.ht_capacity[0] = buckets
    check(plan, acc, tuning=t, label="buckets=%d" % buckets)


@pytest.mark.parametrize("probe", [0, 1, 255, 3071, 3072, 3073, 40000])
@pytest.mark.parametrize("plan", ["c2_pushdown", "c2_both", "c2_batch"])
def test_gather(probe, plan):
    import numpy as np
    from dogqc_amd import batching
    acc = workloadAcc("c2", {"build": max(1, probe // 8), "probe": probe}, seed=probe + 7)
    if plan == "c2_batch":
        if not probe:
            return
        acc = batching.withBatch(acc, {t: np.array([max(1, n // 2), n], dtype=np.int64)
                                       for t, n in (("build", max(1, probe // 8)), ("probe", probe))})
    for grid, threshold, longList in ((0, 0, 0), (3, 1, 1), (3, 64, 20), (1, 33, 100000)):
        t = rt.newTuning()
        for i in range(rt.MAX_PIPES):
            t.grid[i], t.refill_threshold[i], t.split_threshold[i] = grid, threshold, longList
        check(plan, acc, tuning=t, label="probe=%d grid=%d threshold=%d split=%d" % (probe, grid, threshold, longList))
