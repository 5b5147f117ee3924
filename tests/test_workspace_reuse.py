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
