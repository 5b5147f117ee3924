"""Group-bys on probe-row keys inside a per-lane match loop: accumulated in
registers over a row's matches, one update per row.  Rows without a match,
with one, and with many; outer joins' null rows."""
import numpy as np
import pytest

from dogqc_amd import planlib
from tests.test_gpu_parity import check


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [0, 1, 63, 64, 65, 3000])
@pytest.mark.parametrize("nu", [0, 1, 70, 900])
@pytest.mark.parametrize("dup", [False, True])
def test_per_probe_row(nt, nu, dup):
    acc = planlib.featureData(nt, nu, seed=nt + nu)
    if dup:     # every build row in one list
        acc.data[("u", "u_grp")] = np.full(nu, 7, dtype=np.int32)
    for plan in ("f_outer", "f_join_string", "f_join_multi", "f_outer_project"):
        check(plan, acc, label="nt=%d nu=%d dup=%s" % (nt, nu, dup))
