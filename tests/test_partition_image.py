"""Partitioned group-by with each partition's slot range held in LDS."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

from dogqc_amd import plancache, planlib, runtime as rt
from tests.test_gpu_parity import check, module

M64 = (1 << 64) - 1


@pytest.fixture(scope="module")
def ranges(tmp_path_factory):
    """The header's own hash and range functions, compiled for the host."""
    text = open(os.path.join(plancache.CSRC, "dqc_device.h")).read()
    src = "#include <cmath>\n#include <cstdint>\n#define DQC_DEVICE_INLINE static inline\n"
    for name in ("mix64", "slot_of", "part_of", "part_lo", "part_home", "part_slots"):
        src += re.search(r"^(?:DQC_DEVICE_INLINE|inline) \w+ %s\([^{]*\{(?:[^\n]*\}\n|.*?^\}\n)" % name, text, re.M | re.S).group(0)
    src += """extern "C" void place(const uint64_t* h, long n, uint32_t bits, uint32_t cap, uint32_t* out) {
    for (long i = 0; i < n; ++i) {
        const uint32_t p = part_of(h[i], bits), lo = part_lo(p, bits, cap), hi = part_lo(p + 1u, bits, cap);
        out[4 * i] = p; out[4 * i + 1] = lo; out[4 * i + 2] = hi; out[4 * i + 3] = part_home(h[i], cap, hi);
    }
}
extern "C" void hashes(const uint64_t* k, long n, uint64_t* h) { for (long i = 0; i < n; ++i) h[i] = mix64(k[i]); }
extern "C" uint64_t slots(uint64_t cap, uint32_t np) { return part_slots(cap, np); }
"""
    d = tmp_path_factory.mktemp("ranges")
    (d / "r.cpp").write_text(src)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", str(d / "r.cpp"), "-o", str(d / "r.so")], check=True)
    lib = ctypes.CDLL(str(d / "r.so"))
    lib.slots.restype = ctypes.c_uint64
    lib.slots.argtypes = [ctypes.c_uint64, ctypes.c_uint32]
    return lib


def place(lib, h, bits, cap):
    out = np.zeros((len(h), 4), dtype=np.uint32)
    lib.place(h.ctypes.data_as(ctypes.c_void_p), ctypes.c_long(len(h)), ctypes.c_uint32(bits), ctypes.c_uint32(cap),
              out.ctypes.data_as(ctypes.c_void_p))
    return out.T


def test_ranges_hold_their_home_slots(ranges):
    """Every hash's home slot lies in its partition's range, and the ranges
    cut the table."""
    rng = np.random.default_rng(3)
    for bits in (0, 1, 5, 10):
        np_ = 1 << bits
        for cap in {np_, np_ + 1, 2 * np_ - 1, 1000003, 3 * np_ + 7, (1 << 32) - 2}:
            if cap < np_:
                continue
            edges = [((p << (64 - bits)) + d) & M64 for p in range(np_ + 1) for d in (0, 1, -1)]
            h = np.concatenate([rng.integers(0, M64, 500, dtype=np.uint64), np.array(edges, dtype=np.uint64)])
            part, lo, hi, home = place(ranges, h, bits, cap)
            assert (part < np_).all() and (lo <= home).all() and (home < hi).all()
            byPart = {int(p): (int(a), int(b)) for p, a, b in zip(part, lo, hi)}
            cuts = [byPart[p] for p in range(np_)]
            assert cuts[0][0] == 0 and cuts[-1][1] == cap and all(a[1] == b[0] for a, b in zip(cuts, cuts[1:]))


@pytest.mark.parametrize("parts", [2, 256, 1024])
@pytest.mark.parametrize("keys", [1, 300, 2049, 2100, 2600, 3000, 4000, 6000, 20000, 300000])
def test_a_partitions_groups_fit_its_range(keys, parts, ranges):
    """A table sized for exactly its groups, as partitions' ranges of the
    slots it then has: no range gets more groups than slots."""
    for cap in (keys, 2 * keys):
        slots = ranges.slots(cap, parts)
        assert slots >= cap and slots % parts == 0
        for k in [np.arange(keys, dtype=np.uint64)] + [np.random.default_rng(s).choice(1 << 40, keys, replace=False)
                                                       .astype(np.uint64) for s in range(3)]:
            h = np.zeros(keys, dtype=np.uint64)
            ranges.hashes((k + np.uint64(1)).ctypes.data_as(ctypes.c_void_p), ctypes.c_long(keys),
                          h.ctypes.data_as(ctypes.c_void_p))
            part, lo, hi, _ = place(ranges, h, parts.bit_length() - 1, slots)
            assert (hi - lo == slots // parts).all()
            assert np.bincount(part).max() <= slots // parts, (keys, cap)


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
        # a table of two slots a group, or partitioned with a slot a group, holds
        # them: not enlarged (a retry may be for the result's rows)
        if cap == 0 or cap >= 2 * keys or (cap >= keys and 2 <= parts <= cap):
            assert t.ht_capacity[0] == cap


@pytest.mark.gpu
@pytest.mark.parametrize("keys", [2049, 2100, 2600, 3000, 4000, 6000])
def test_learned_sizes_hold_the_groups(keys):
    """Sizes that Feedback learned: neither a run nor an enqueue at them
    overflows, with as many partitions as the plan chooses by itself."""
    acc = accessor(70001, keys, False)
    mod = module("f_groupby_int64")
    inputs = rt.BoundInputs(mod, acc)
    fb = rt.Feedback()
    rt.run(mod, inputs, feedback=fb).release()
    t = rt.newTuning()
    fb.apply(mod, inputs, t)
    # (the key -1 has the extra slot)
    assert 2 * (keys - 1) <= t.ht_capacity[0] <= 2 * keys
    _, retries = check("f_groupby_int64", acc, tuning=t, label="learned, keys=%d" % keys)
    assert retries == 0 and t.ht_capacity[0] <= 2 * keys
    ws, stream = rt.DeviceBuffer(int(rt.layout(mod, inputs, t).ws_bytes)), rt.Stream()
    rt.enqueue(mod, inputs, t, ws, stream)
    stream.sync()
    ex = rt.view(mod, inputs, t, ws)
    assert ex.res.status.flags == 0 and ex.count == keys
