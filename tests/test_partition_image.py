"""Partitioned group-by with each partition's slot range held in LDS."""
import numpy as np
import pytest

from dogqc_amd import planlib, runtime as rt
from tests.test_gpu_parity import check

M64 = (1 << 64) - 1


def test_ranges_hold_their_home_slots():
    """dqc::part_of, part_lo, part_home and slot_of: every hash's home slot
    lies in its partition's range, and the ranges cut the table."""
    rng = np.random.default_rng(3)
    for bits in (0, 1, 5, 10):
        np_ = 1 << bits
        for cap in {np_, np_ + 1, 2 * np_ - 1, 1000003, 3 * np_ + 7, (1 << 32) - 2}:
            if cap < np_:
                continue
            lo = [(p * cap) >> bits for p in range(np_ + 1)]
            assert lo[0] == 0 and lo[-1] == cap and all(b > a for a, b in zip(lo, lo[1:]))
            edges = [(p << (64 - bits)) + d for p in range(min(np_, 40)) for d in (0, 1)] + [
                ((p + 1) << (64 - bits)) - 1 for p in range(min(np_, 40))]
            for h in [int(x) for x in rng.integers(0, M64, 500, dtype=np.uint64)] + edges:
                h &= M64
                part = (h >> 32) >> (32 - bits)
                slot = ((h >> 32) * cap) >> 32
                assert part < np_ and lo[part] <= slot <= lo[part + 1]      # the upper end by rounding only
                home = slot if slot < lo[part + 1] else lo[part + 1] - 1
                assert lo[part] <= home < lo[part + 1]


def accessor(n, keys, skew):
    """t_big / 2^30 takes `keys` values from -1 on (-1: the tag-0 key of the
    extra slot); skewed: nine rows in ten hold one of them."""
    acc = planlib.featureData(n, 10, seed=n)
    k = np.arange(n, dtype=np.int64) % keys - 1
    if skew:
        k[np.arange(n) % 10 != 0] = min(keys - 1, 5) - 1
    acc.data[("t", "t_big")] = k * (1 << 30) - (k < 0) * 5
    return acc


@pytest.mark.gpu
@pytest.mark.parametrize("n,keys", [(1, 1), (300, 300), (5000, 2050), (70001, 4000), (70001, 9)])
@pytest.mark.parametrize("parts", [0, 2, 256, 1024])
@pytest.mark.parametrize("skew", [False, True])
def test_image(n, keys, parts, skew):
    acc = accessor(n, keys, skew)
    for cap in (0, keys, keys + 3, 3 * keys + 1, 1024, 40000):
        t = rt.newTuning()
        t.part_agg, t.ht_capacity[0] = parts, cap
        check("f_groupby_int64", acc, tuning=t, label="n=%d keys=%d parts=%d cap=%d" % (n, keys, parts, cap))
