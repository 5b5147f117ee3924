"""Multimap directory scan at tile and look-back edges; push-down probes that
gather their rows first, at trip edges, thresholds and split list lengths."""
import numpy as np
import pytest

from dogqc_amd import planlib, runtime as rt
from tests.test_gpu_parity import check, workloadAcc


# 4096 buckets a tile; 64 tiles a look-back step
@pytest.mark.gpu
@pytest.mark.parametrize("buckets", [1, 63, 4095, 4096, 4097, 64 * 4096, 64 * 4096 + 1, 200 * 4096 + 17])
@pytest.mark.parametrize("plan", ["c2_none", "c2_pushdown"])
def test_directory_scan(buckets, plan):
    acc = workloadAcc("c2", {"build": 3000, "probe": 5000}, seed=buckets)
    t = rt.newTuning()
    t.ht_capacity[0] = buckets
    check(plan, acc, tuning=t, label="buckets=%d" % buckets)


@pytest.mark.gpu
@pytest.mark.parametrize("probe", [0, 1, 255, 3071, 3072, 3073, 40000])
@pytest.mark.parametrize("plan", ["c2_pushdown", "c2_both", "c2_batch"])
def test_gather(probe, plan):
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


def test_any_source_gathers():
    """Several rows per thread and the gathering probe (or the lane refill)
    go together, whatever the pipeline reads: here a group table."""
    for plan in ("f_group_probe_pushdown", "f_group_refill"):
        pipe = next(p for p in planlib.translate(plan).program.pipes if p.name.startswith("krnl_aggregation"))
        assert pipe.frontU > 1 and pipe.U == 1
        assert pipe.drains if plan == "f_group_probe_pushdown" else pipe.refillPoints


# the group table's slots around a trip of the grid; with and without long
# lists (the filter keeps groups of more than 42 rows)
@pytest.mark.gpu
@pytest.mark.parametrize("groups", [1, 63, 100, 511, 1023, 1025, 1600])
@pytest.mark.parametrize("plan", ["f_group_probe_pushdown", "f_group_refill"])
def test_group_table_source(groups, plan):
    acc = planlib.featureData(64 * groups, 700, seed=groups)
    n = np.arange(64 * groups)
    acc.data[("t", "t_grp")] = (np.where(n % 3 == 0, 7 % groups, n % groups) - 1).astype(np.int32)
    for grid, threshold, longList in ((0, 0, 0), (1, 1, 1), (1, 64, 3), (3, 0, 100000)):
        t = rt.newTuning()
        for i in range(rt.MAX_PIPES):
            t.grid[i], t.refill_threshold[i], t.split_threshold[i] = grid, threshold, longList
        t.ht_capacity[1] = 2 * groups + 1
        check(plan, acc, tuning=t, label="groups=%d grid=%d threshold=%d" % (groups, grid, threshold))
