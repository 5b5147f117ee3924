"""Unique join tables at the loads and sizes where a probe's window meets the
table's end, wraps, or is full: capacities of exactly the keys and a few more."""
import pytest

from dogqc_amd import planlib, runtime as rt
from tests.test_gpu_parity import check, module, workloadAcc

PLANS = ["c1", "f_join_neg", "f_anti_neg", "f_join_packed", "f_join_unique", "tpch5"]


def accessor(plan, size):
    if plan == "c1":
        return workloadAcc("c1", {"dim": 5 * size, "fact": 400}, seed=size)
    if plan == "tpch5":
        from dogqc_amd import tpch
        from dogqc_amd.dbio import MemoryAccessor
        return MemoryAccessor(tpch.generate(0.0005 * size, seed=size))
    return planlib.featureData(300, size, seed=size)


@pytest.mark.gpu
@pytest.mark.parametrize("plan", PLANS)
@pytest.mark.parametrize("size", [1, 2, 3, 4, 5, 9, 60])
def test_tight_tables(plan, size):
    acc = accessor(plan, size)
    mod = module(plan)
    inputs = rt.BoundInputs(mod, acc)
    fb = rt.Feedback()
    rt.run(mod, inputs, rt.newTuning(), feedback=fb).release()
    rec = fb.records[fb.key(mod)]
    for extra in (0, 1, 2, 3, 5):
        t = rt.newTuning()
        for i, kind in enumerate(rec["kinds"]):
            if kind == "unique":
                t.ht_capacity[i] = max(1, rec["fill"][i] + extra)
        check(plan, acc, tuning=t, label="size=%d extra=%d" % (size, extra))
