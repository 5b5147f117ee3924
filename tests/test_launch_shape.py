"""Row-to-thread mapping of pipelines with several rows per thread: a table of
at least one full trip of the grid is walked in tiles, a smaller one in steps
of the whole grid, and both have to reach every row exactly once."""
import ctypes
import re
import subprocess

import numpy as np
import pytest

import dogqc_amd.scalarAlgebra as scal
from dogqc_amd import planlib, runtime as rt
from dogqc_amd.relationalAlgebra import Reduction
from dogqc_amd.types import Type
from tests.test_gpu_parity import check, workloadAcc

GRID = 3


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    """Rows in the order that the loop of a generated kernel assigns them: its
    own statements (Pipeline.render), compiled for the host."""
    built = {}

    def rows(U, n, grid):
        if U not in built:
            with planlib.knobs(rowsPerThread=U):
                comp = planlib.translate("c1", rowsPerThread=U)
            pipe = comp.program.pipes[0]
            assert pipe.frontU == U
            body = comp.source[comp.source.index(" %s(const" % pipe.name):]
            own = [ln.strip() for ln in body[:body.index("active[u] = more")].splitlines()]
            head = [ln for ln in own if ln.startswith(("const bool tiled", "const int64_t step"))]
            loop = [ln for ln in own if ln.startswith("for (int64_t base")]
            row = [ln for ln in own if ln.startswith("%s[u] = base" % pipe.tid)]
            assert loop and len(loop) == len(row) == 1
            d = tmp_path_factory.mktemp("walk")
            (d / "w.cpp").write_text("""#include <cstdint>
struct dim { uint32_t x; };
extern "C" long walk(int64_t nrows, uint32_t grid, int64_t* out) {
    long n = 0;
    const dim gridDim{grid};
    dim blockIdx{0}, threadIdx{0};
    for (; blockIdx.x < grid; ++blockIdx.x)
        for (threadIdx.x = 0; threadIdx.x < %du; ++threadIdx.x) {
            %s
            %s
                for (int u = 0; u < %d; ++u) {
                    int64_t %s[%d];
                    %s
                    if (%s[u] < nrows) out[n++] = %s[u];
                }
            }
        }
    return n;
}
""" % (pipe.bs, "\n".join(head), loop[0], U, pipe.tid, U, row[0], pipe.tid, pipe.tid))
            subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(d / "w.cpp"), "-o", str(d / "w.so")], check=True)
            built[U] = (ctypes.CDLL(str(d / "w.so")), pipe.bs)
        lib, _ = built[U]
        out = np.zeros(2 * n + 1, dtype=np.int64)
        count = lib.walk(ctypes.c_int64(n), ctypes.c_uint32(grid), out.ctypes.data_as(ctypes.c_void_p))
        return out[:count], built[U][1]
    return rows


@pytest.mark.parametrize("U", [1, 2, 4])
def test_every_row_once(U, walk):
    B = walk(U, 1, 1)[1]
    for grid in (1, 3, 4):
        full = grid * B * U
        for n in {0, 1, B - 1, B, B + 1, full - 1, full, full + 1, 2 * full - 1, 2 * full, 2 * full + B + 1}:
            assert np.array_equal(np.sort(walk(U, n, grid)[0]), np.arange(n)), (U, grid, n)


# one full trip of 3 workgroups x 256 threads x 4 rows is 3072 rows
@pytest.mark.gpu
@pytest.mark.parametrize("plan", ["c0", "c1", "c0_batch"])
@pytest.mark.parametrize("n", [1, 255, 257, 3071, 3072, 3073, 6143, 6145])
def test_edges(plan, n):
    t = rt.newTuning()
    for i in range(rt.MAX_PIPES):
        t.grid[i] = GRID
    if plan == "c0_batch":
        from dogqc_amd import batching
        acc = workloadAcc("c0", {"cfg0": n}, seed=n)
        acc = batching.withBatch(acc, {"cfg0": np.array(sorted({max(1, n // 3), max(1, n // 2), n}), dtype=np.int64)})
    else:
        acc = workloadAcc(plan, {"cfg0": n} if plan == "c0" else {"dim": n, "fact": n + 5}, seed=n)
    check(plan, acc, tuning=t, label="n=%d" % n)


# the LDS table's 16-slot front: fewer groups than it has slots, as many, more,
# and the key (-1, -1) whose 64-bit tag is 0 and bypasses the LDS table
@pytest.mark.gpu
@pytest.mark.parametrize("groups", [1, 2, 13, 16, 17, 60, 128])
@pytest.mark.parametrize("n", [1, 1025, 70001])
def test_front_table(groups, n):
    acc = planlib.featureData(n, 10, seed=groups)
    acc.data[("t", "t_grp")] = (np.arange(n) % groups - 1).astype(np.int32)
    check("f_groupby_64", acc, label="groups=%d n=%d" % (groups, n))
    check("f_groupby_wide", acc, label="groups=%d n=%d" % (groups, n))


# a string filter into a multimap build: the second launch takes the rows
# that passed from the first launch's ranks, tiled and in steps of the grid
@pytest.mark.gpu
@pytest.mark.parametrize("orders", [8, 255, 3071, 3072, 3073])
@pytest.mark.parametrize("grid", [0, GRID])
def test_ranked_rows(orders, grid):
    from dogqc_amd import tpch
    from dogqc_amd.dbio import MemoryAccessor
    acc = MemoryAccessor(tpch.generate(orders / 1.5e6, seed=orders))
    t = rt.newTuning()
    for i in range(rt.MAX_PIPES):
        t.grid[i] = grid
    for q in ("tpch13", "tpch16"):
        check(q, acc, tuning=t, label="orders=%d" % orders)


# lane refill behind several rows per thread, with the refill above a filtered
# join placed between the filter and the probe: trips' edges, thresholds, and
# the filter off, in LDS and in device memory
@pytest.mark.gpu
@pytest.mark.parametrize("plan", ["c1_refill", "c3_refill", "tpch10", "f_like_project_refill"])
@pytest.mark.parametrize("n", [1, 257, 3071, 3073, 9000])
def test_refill_front(plan, n):
    from dogqc_amd import tpch
    from dogqc_amd.dbio import MemoryAccessor
    if plan == "tpch10":
        acc = MemoryAccessor(tpch.generate(n / 6.0e6, seed=n))
    elif plan == "c1_refill":
        acc = workloadAcc("c1", {"dim": max(1, n // 4), "fact": n}, seed=n)
    elif plan == "c3_refill":
        acc = workloadAcc("c3", {"sales": n, "item": max(1, n // 20), "cust": max(1, n // 50)}, seed=n)
    else:
        acc = planlib.featureData(n, 10, seed=n)
    for grid, threshold, jf in ((0, 0, 0), (GRID, 1, 0), (GRID, 64, -1), (GRID, 0, 32), (1, 0, 1024), (5000, 64, 0)):
        t = rt.newTuning()
        t.join_filter = jf
        for i in range(rt.MAX_PIPES):
            t.grid[i], t.refill_threshold[i] = grid, threshold
        check(plan, acc, tuning=t, label="n=%d grid=%d threshold=%d filter=%d" % (n, grid, threshold, jf))


def test_default_filter_is_held_in_lds(tmp_path):
    """A filter of a size the plan was translated with goes to LDS like one
    the tuning asks for; the size chosen from the key count does not.  (The
    generated host code's own statements, compiled for the host.)"""
    def words(default, request):
        alg, p, cfg, opts = planlib.build("c3_refill", planlib.emptyAccessor("c3_refill"))
        plan = alg.resolveAlgebraPlan(p, cfg)
        with planlib.knobs(joinFilter=default):
            comp = planlib.HipCompiler(alg, "gfx950", planlib.CType.FP64)
            comp.setBuffers(opts["buffers"])
            comp.gencode(alg.translateToCompilerPlan(plan, comp))
        size = re.search(r"\{ const int32_t req = .*?L\.bfw\[2\] = w; \}", comp.source, re.S).group(0)
        held = re.search(r"L\.bfp\[\d+\] = [^;]*\? L\.bfw\[2\] : 0u;", comp.source).group(0)
        helpers = "".join(re.search(r"static inline uint32_t pow2%s\(.*\n" % f, comp.source).group(0)
                          for f in ("floor", "ceil"))
        (tmp_path / "w.cpp").write_text(
            "#include <algorithm>\n#include <cstdint>\n#include <cstdio>\n" + helpers +
            "static uint64_t maxLds() { return 163840; }\n"
            "int main() { struct { uint32_t bfw[4], bfp[4]; int64_t htcap[4]; } L = {}; L.htcap[2] = 60000;\n"
            "struct { int32_t join_filter; } T = {%d}, *t = &T;\n%s\n%s\n"
            "printf(\"%%u %%u\\n\", L.bfw[2], L.bfp[0] + L.bfp[1] + L.bfp[2] + L.bfp[3]); }\n" % (request, size, held))
        subprocess.run(["g++", "-std=c++17", "-w", str(tmp_path / "w.cpp"), "-o", str(tmp_path / "w")], check=True)
        return [int(x) for x in subprocess.run([str(tmp_path / "w")], stdout=subprocess.PIPE, check=True).stdout.split()]

    assert words(32, 0) == words(0, 32) == [8192, 8192]
    assert words(32, -1) == words(0, -1) == [0, 0]
    assert words(32, 64) == [16384, 16384]
    assert words(0, 0) == [16384, 0]
    assert words(2048, 0) == [524288, 0]


@pytest.mark.parametrize("plan", ["c2_pushdown", "c2_both", "c3_refill", "f_like_project_refill", "tpch3", "tpch5",
                                  "tpch7", "tpch8", "tpch9", "tpch10", "tpch14", "tpch19"])
@pytest.mark.parametrize("budget", [80 << 10, 40 << 10, 16 << 10, 0])
def test_queue_stays_in_its_lds(plan, budget, monkeypatch):
    """A queue holds no more per row than the bound that chose the rows per
    thread, so it keeps to its share of LDS (or to one row per thread)."""
    from dogqc_amd import hipTranslator as H
    monkeypatch.setattr(H, "QUEUE_LDS", budget)
    bounds, bound = [], H.queuedBytes
    monkeypatch.setattr(H, "queuedBytes", lambda t: bounds.append(bound(t)) or bounds[-1])
    for pipe in planlib.translate(plan).program.pipes:
        if not (pipe.refillPoints or pipe.drains):
            continue
        pipe.staticLds = [d for d in pipe.staticLds if d.split()[2].startswith(("rq", "pg"))]
        rows = (pipe.bs // 64) * 64 * (pipe.frontU + 1)
        assert H.staticLdsBytes(pipe) <= rows * sum(bounds), (plan, bounds)
        assert pipe.frontU == 1 or rows * max(bounds) <= budget


def _twoRefills(alg, A, C):
    """A group table through two lane refills into a result of 20 bytes a row."""
    p = alg.projection(["t_id", "g", "m"],
                       alg.map("m", scal.MulExpr(A("g"), C("2", Type.DOUBLE)),
                               alg.aggregation(["t_id"], [(Reduction.MIN, "t_val", "g")], alg.scan("t"))))
    return p, {}, [2, 4]


def _stringJoin(alg, A, C):
    """A selective unique join on a string, a refill right above it and one
    more below the result: the first queue before the probe would hold the key."""
    p = alg.projection(["u_id", "u_w", "u_grp"],
                       alg.selection(scal.LargerExpr(A("u_w"), C("1.5", Type.DOUBLE)),
                                     alg.selection(scal.LargerExpr(A("u_grp"), C("2", Type.INT)),
                                                   alg.join(("u_name", "t_txt"), alg.scan("u"), alg.scan("t")))))
    return p, {3: {"multimatch": False, "selectivity": 0.1}}, [3, 5]


def _wideProbe(alg, A, C):
    """A push-down probe that few rows reach, of rows with many strings: it
    gathers them where their queue fits."""
    node, cols = alg.scan("t"), ["s%d" % k for k in range(8)]
    for k, c in enumerate(cols):
        node = alg.map(c, scal.SubstringExpr(A("t_txt"), C(str(k + 1), Type.INT), C("3", Type.INT)), node)
    node = alg.selection(scal.LargerExpr(A("t_id"), C("2", Type.INT)), node)
    node = alg.join(("u_grp", "t_grp"), alg.scan("u"), node)
    for a, b in zip(cols, cols[1:]):
        node = alg.selection(scal.NotExpr(scal.EqualsExpr(A(a), A(b))), node)
    return alg.projection(["u_id", "s0"], node), {10: {"selectivity": 0.1}, 12: {"multimatch": True}}, []


@pytest.mark.parametrize("plan", [_twoRefills, _stringJoin, _wideProbe])
@pytest.mark.parametrize("block,rows", [(256, 4), (256, 8), (512, 4), (1024, 1), (1024, 4)])
def test_queues_leave_lds_to_the_operators_above(plan, block, rows):
    """All of a pipeline's static LDS fits a CU: the rows per thread, and the
    place of a refill at a filtered join, leave room for what follows."""
    from dogqc_amd import hipTranslator as H
    alg = planlib.RelationalAlgebra(planlib.featureEmpty())
    p, cfg, buffers = plan(alg, planlib._A, planlib._C)
    resolved = alg.resolveAlgebraPlan(p, cfg)
    with planlib.knobs(block=block, rowsPerThread=rows, pushdown=plan is _wideProbe):
        comp = H.HipCompiler(alg, "gfx950", planlib.CType.FP64)
        comp.setBuffers(buffers)
        comp.gencode(alg.translateToCompilerPlan(resolved, comp))
    assert block > 256 or any(q.refillPoints or q.drains for q in comp.program.pipes)
    assert max(H.staticLdsBytes(q) for q in comp.program.pipes) <= 160 << 10


def test_join_builds_take_a_row_per_thread():
    """A pipeline that ends in inserts into a join table is launched on four
    times the workgroups of the others."""
    src = planlib.translate("c1").source
    calls = re.findall(r"gridFor\(t->grid[^;]*?,\s*(\d+),\s*(\d+),\s*(\d+),\s*(\d+)\);", src)
    (_, build, _, spread), others = [int(x) for x in calls[0]], [[int(x) for x in c] for c in calls[1:]]
    assert others and spread == build and all(build == 4 * perCu for _, perCu, _, _ in others)


# the build's grid ends at 256 CUs x 32 workgroups x 256 rows
@pytest.mark.gpu
@pytest.mark.parametrize("n", [2048 * 256 + 1, 8192 * 256 - 1, 8192 * 256 + 1, 8192 * 1024 + 257])
def test_join_build_grid(n):
    check("c1", workloadAcc("c1", {"dim": n, "fact": 1 << 16}, seed=n % 97), label="dim=%d" % n)


def test_a_programs_default_grid_is_taken(monkeypatch):
    """KernelCall.defaultGridSize holds for every pipeline that the tuning
    gives no grid, also those whose grid follows from groups or queues."""
    from dogqc_amd.kernel import KernelCall
    for plan in ("c0", "c1_refill", "c2_pushdown", "tpch1"):
        monkeypatch.setattr(KernelCall, "defaultGridSize", 0)
        chosen = planlib.translate(plan).source
        monkeypatch.setattr(KernelCall, "defaultGridSize", 7)
        asked = planlib.translate(plan).source
        assert "] <= 0) g = " in chosen and "] <= 0) g = " not in asked, plan
        assert "] : 7, " in asked and "] : 0, " not in asked


def test_scalar_registers_of_large_workgroups():
    """Large workgroups that share a CU are limited to 80 scalar registers;
    with few groups, or static LDS of more than half a CU, they have it alone."""
    from dogqc_amd import autotune
    from dogqc_amd.hipTranslator import staticLdsBytes
    comp = autotune.translateVariant("tpch2", 1024, 1)
    alone = [staticLdsBytes(p) > 80 << 10 for p in comp.program.pipes]
    assert any(alone) and not all(alone)
    for p, one in zip(comp.program.pipes, alone):
        assert ("amdgpu_num_sgpr(80))) %s(" % p.name in comp.source) == (not one and p.bs >= 512 and not p.fewGroups)
    few, many, small = planlib.translate("tpch1").source, planlib.translate("tpch18").source, planlib.translate("c1").source
    assert "__launch_bounds__(1024) krnl_lineitem1(" in few
    assert "__launch_bounds__(1024) __attribute__((amdgpu_num_sgpr(80))) krnl_lineitem1(" in many
    assert "amdgpu_num_sgpr" not in small
