"""Workspaces that wait for the next run: results kept alive keep their own
memory, and threads with streams of their own do not share any."""
import threading

import pytest

from dogqc_amd import runtime as rt, runner
from tests.helpers import assertSameResult, toleranceColumns
from tests.test_gpu_parity import module, oracleFor, workloadAcc

pytestmark = pytest.mark.gpu


def start(plan, rows, seed):
    acc = workloadAcc(plan, rows, seed)
    mod = module(plan)
    return acc, mod, rt.BoundInputs(mod, acc), oracleFor(plan, acc)


def verify(acc, mod, ex, expected, label):
    want, plan = expected
    assertSameResult(runner.resultColumns(mod, ex, acc), want, toleranceColumns(plan), label=label)


def test_kept_results_survive_later_runs():
    a = start("c1", {"dim": 4000, "fact": 20000}, 1)
    b = start("c1", {"dim": 3000, "fact": 50000}, 2)
    first = rt.run(a[1], a[2])
    for k in range(3):
        ex = rt.run(b[1], b[2])
        assert ex.res.ws != first.res.ws
        verify(b[0], b[1], ex, b[3], "run %d" % k)
        ex.release()
    verify(a[0], a[1], first, a[3], "kept result")
    first.release()
    again = rt.run(b[1], b[2])
    verify(b[0], b[1], again, b[3], "after release")
    again.release()


def test_a_larger_run_after_a_smaller():
    small, large = start("c1", {"dim": 50, "fact": 100}, 3), start("c0", {"cfg0": 300000}, 4)
    wide = start("c1", {"dim": 60000, "fact": 1000}, 5)
    for s in (small, wide, small, large, wide):
        ex = rt.run(s[1], s[2])
        verify(s[0], s[1], ex, s[3], "mixed sizes")
        ex.release()


def test_a_kept_small_result_leaves_the_large_block():
    small, large = start("c1", {"dim": 50, "fact": 100}, 6), start("c1", {"dim": 2400000, "fact": 1000}, 7)
    rt.trimWorkspaces()
    ex = rt.run(large[1], large[2])
    block = ex.res.ws
    assert ex.res.ws_bytes > (5 << 20)
    ex.release()
    kept = rt.run(small[1], small[2])
    assert kept.res.ws != block
    ex = rt.run(large[1], large[2])
    assert ex.res.ws == block
    verify(large[0], large[1], ex, large[3], "large again")
    ex.release()
    verify(small[0], small[1], kept, small[3], "kept small")
    kept.release()


def freeBytes():
    free, total = rt.C.c_size_t(), rt.C.c_size_t()
    assert rt.lib().hipMemGetInfo(rt.C.byref(free), rt.C.byref(total)) == 0
    return free.value


def test_trim_gives_the_memory_back():
    job = start("c0", {"cfg0": 1000}, 8)
    t = rt.newTuning()
    t.result_capacity = 8 << 20         # some 700 MB of result columns
    before = freeBytes()
    ex = rt.run(job[1], job[2], t)
    size = ex.res.ws_bytes
    verify(job[0], job[1], ex, job[3], "large result")
    ex.release()
    assert before - freeBytes() >= size // 2
    rt.trimWorkspaces()
    assert before - freeBytes() < size // 2


def test_a_workspace_freed_by_hand_is_forgotten():
    """dqc_free on a result's workspace, as dqc_query_release did at first:
    a smaller allocation that gets the address is not taken for it."""
    job = start("c1", {"dim": 600000, "fact": 1000}, 9)
    rt.trimWorkspaces()
    ex = rt.run(job[1], job[2])
    rt.check(rt.lib().dqc_free(ex.res.ws), "dqc_free")
    ex.res.ws = None
    other = rt.DeviceBuffer(4096)
    res = rt.QueryResult()
    res.ws, res.ws_bytes = other.ptr.value, 4096
    rt.check(rt.lib().dqc_query_release(rt.C.byref(res)), "dqc_query_release")
    other.ptr = rt.C.c_void_p()
    ex = rt.run(job[1], job[2])
    verify(job[0], job[1], ex, job[3], "after dqc_free")
    ex.release()


def test_threads():
    jobs = [start("c1", {"dim": 1000 * (k + 1), "fact": 30000}, 10 + k) for k in range(4)]
    failures = []

    def work(job):
        try:
            stream = rt.Stream()
            for _ in range(20):
                ex = rt.run(job[1], job[2], stream=stream)
                verify(job[0], job[1], ex, job[3], "thread")
                ex.release()
        except BaseException as e:      # reported by the test's own thread
            failures.append(e)

    threads = [threading.Thread(target=work, args=(j,)) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures[0]
