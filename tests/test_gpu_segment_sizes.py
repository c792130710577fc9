"""Persistent segmented kernels with 8-bit digits: bit-exact against the oracle
at the edges of their size classes (one lane per key, one wave with 2, 4, 8
keys per lane, one workgroup with 2, 4, 6, 8, 12, 16 per thread), for each
value class, and which kernels take segments between 4097 keys and a
workgroup's tile."""
import numpy as np
import pytest

from mgpu_old_amd import workloads
from gpu_helpers import GpuSort, make_engine

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047,
         2048, 2049, 3071, 3072, 3073, 4095, 4096, 4097, 6143, 6144, 6145, 8191, 8192]


@pytest.fixture(scope="module")
def engine():
    eng = make_engine()
    yield eng
    eng.close()


def _starts(sizes):
    return np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)


def _keys(starts, seed):
    """Uniform keys, with equal, all-ones and few-valued segments among them."""
    keys = workloads.uniform_keys(int(starts[-1]), seed=seed)
    for i in range(len(starts) - 1):
        part = keys[starts[i]:starts[i + 1]]
        if i % 5 == 1:
            part[:] = 0xFFFFFFFF
        elif i % 5 == 2:
            part &= np.uint32(0x01010101)
        elif i % 5 == 3:
            part |= np.uint32(0xFFFFFF00)
    return keys


def _run(engine, oracle, sizes, vc, fb, eb, seed):
    starts = _starts(sizes)
    keys = _keys(starts, seed)
    vals = [workloads.uniform_keys(len(keys), seed=seed + 1 + j) for j in range(max(vc, 0))]
    g = GpuSort(keys, vals, value_count=vc, first_bit=fb, end_bit=eb)
    import torch
    torch.cuda.synchronize()
    engine.enable_timing(True)
    engine.read_timing()
    engine.sort_segmented(g.data, starts)
    torch.cuda.synchronize()
    names = set(engine.read_timing())
    engine.enable_timing(False)
    engine.check_device()
    out_k, out_v = g.keys(), g.values()
    for i in range(len(sizes)):
        a, b = int(starts[i]), int(starts[i + 1])
        rk, rv = oracle.stable_sort(keys[a:b], [v[a:b] for v in vals], value_count=vc,
                                    first_bit=fb, end_bit=eb)
        assert np.array_equal(out_k[a:b], rk), f"segment {i} (n={b - a}) keys differ"
        for j, (o, r) in enumerate(zip(out_v, rv)):
            assert np.array_equal(o[a:b], r), f"segment {i} (n={b - a}) values[{j}] differ"
    return names


# Three copies of each size in turn: every wave takes several small segments.
@pytest.mark.parametrize("vc", [-1, 0, 1, 2, 6])
@pytest.mark.parametrize("fb,eb", [(0, 32), (3, 20), (8, 32), (31, 32)])
def test_size_class_edges(engine, oracle, vc, fb, eb):
    _run(engine, oracle, SIZES * 3, vc, fb, eb, seed=71)


@pytest.mark.parametrize("vc", [-1, 1])
def test_many_small_segments(engine, oracle, vc):
    """More small segments than waves of the grid: the reads ahead of a wave's
    sorts, up to the end of the list."""
    rng = np.random.default_rng(5)
    _run(engine, oracle, list(rng.integers(1, 90, 9001)), vc, 0, 32, seed=73)


@pytest.mark.parametrize("variant", [None, "r8i16", "r7i8"])
def test_many_workgroup_segments(engine, oracle, variant, monkeypatch):
    """More workgroup segments than workgroups: drawn from the cursors, which
    every launch leaves as it found them."""
    if variant:
        monkeypatch.setenv("MGPUSORT_SEG_VARIANT", variant)
    rng = np.random.default_rng(6)
    for seed in (75, 76):
        _run(engine, oracle, list(rng.integers(1025, 1200, 2101)), 1, 0, 32, seed=seed)


@pytest.mark.parametrize("sizes,device_wide", [
    ([8192, 4097, 100], False),
    ([8192, 8193, 100], True),          # longer segments hold more keys
    ([8192, 4097, 8193, 100], False),   # and here fewer
    ([4096, 9000], True),
])
def test_route_above_4096(engine, oracle, sizes, device_wide):
    names = _run(engine, oracle, sizes, 1, 0, 32, seed=79)
    wide = 8193 in sizes or 9000 in sizes
    assert any("mgpu_multi" in k for k in names) == wide, names
    # 8192 and 4097 keys: a workgroup each (16 keys per thread), or with the rest.
    in_tile = any("_r8_i16_" in k for k in names)
    assert in_tile == (not device_wide), names
