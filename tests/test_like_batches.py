"""LIKE literals at every place a search batch (56 start positions of aligned
words) can begin, end or be crossed, in strings of up to three batches."""
from collections import OrderedDict

import numpy as np
import pytest

from dogqc_amd import planlib
from tests.test_gpu_parity import check

# literals of f_like_patterns: 2 bytes, 7, 8 and 13 bytes, and near misses
LITERALS = [b"ha", b"lpha g", b"charlie delta", b"charlie delt", b"juliet juliet", b"o", b"ec-ho", b"a-a-a"]


@pytest.mark.gpu
@pytest.mark.parametrize("lit", LITERALS, ids=lambda b: b.decode().replace(" ", "_"))
def test_every_offset(lit):
    strs = []
    for off in range(0, 130):
        for tail in (0, 1, 7, 60):
            strs.append(b"x" * off + lit + b"y" * tail)
        strs.append(b"x" * off + lit[:-1])          # cut at the end of the string
    acc = planlib.featureData(len(strs), 10, seed=len(lit))
    lens = np.array([len(s) for s in strs], dtype=np.uint64)
    offs = np.zeros(len(strs) + 1, dtype=np.uint64)
    np.cumsum(lens, out=offs[1:])
    acc.data[("t", "t_txt")] = (offs, np.frombuffer(b"".join(strs), dtype=np.uint8))
    acc.data[("t", "t_cat")] = (np.arange(len(strs)) % 100).astype(np.int8)
    check("f_like_patterns", acc, label=repr(lit))
