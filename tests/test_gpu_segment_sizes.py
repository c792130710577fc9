"""Persistent segmented kernels with 8-bit digits: bit-exact against the oracle
at the edges of their size classes (one lane per key, one wave with 2, 4, 8
keys per lane, one workgroup with 2, 4, 6, 8, 12, 16 per thread), for each
value class; which kernels take segments above 4096 keys; and device-wide
segments that one scatter sends to buckets."""
import numpy as np
import pytest

from mgpu_old_amd import workloads
from gpu_helpers import GpuSort, make_engine, to_dev

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


def _check(oracle, keys, vals, vc, starts, g, fb, eb):
    out_k, out_v = g.keys(), g.values()
    for i in range(len(starts) - 1):
        a, b = int(starts[i]), int(starts[i + 1])
        rk, rv = oracle.stable_sort(keys[a:b], [v[a:b] for v in vals], value_count=vc,
                                    first_bit=fb, end_bit=eb)
        assert np.array_equal(out_k[a:b], rk), f"segment {i} (n={b - a}) keys differ"
        for j, (o, r) in enumerate(zip(out_v, rv)):
            assert np.array_equal(o[a:b], r), f"segment {i} (n={b - a}) values[{j}] differ"


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
    _check(oracle, keys, vals, vc, starts, g, fb, eb)
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


@pytest.mark.parametrize("sizes,slots,device_wide", [
    ([8192, 4097, 100], False, False),  # none above the kernels' tile
    ([8193, 8192, 4097, 4096], True, False),
    ([16384, 16385, 4096], True, True),
])
def test_route_above_4096(engine, oracle, sizes, slots, device_wide):
    names = _run(engine, oracle, sizes, 1, 0, 32, seed=79)
    assert any("_slots_" in k for k in names) == slots, names
    assert any("mgpu_multi" in k for k in names) == device_wide, names
    assert any("_r8_i16_" in k for k in names) == (not slots), names


def _spread(kind, n, seed):
    u = workloads.uniform_keys(n, seed=seed)
    if kind == "narrow":  # top digits constant: buckets of a lower digit
        return u >> np.uint32(11)
    if kind == "few":  # 16 values, each in more bins than fit a bucket
        return (u & np.uint32(15)) * np.uint32(0x01010101)
    if kind == "heavy":  # two thirds in one bin: every pass
        return np.where(u % np.uint32(3) == 0, u, u & np.uint32(0xFFFFFF))
    if kind == "equal":
        return np.full(n, 0xFFFFFFFF, dtype=np.uint32)
    return u


KINDS = ["uniform", "narrow", "few", "heavy", "equal"]


@pytest.mark.parametrize("vc", [-1, 0, 1, 2, 6])
@pytest.mark.parametrize("fb,eb", [(0, 32), (5, 26), (0, 16)])  # 4, 3 and (no buckets) 2 passes
def test_buckets(engine, oracle, vc, fb, eb):
    """Device-wide segments of a batch large enough for buckets, each kind of
    keys in segments of each size: 16385 keys, sizes that divide into buckets
    evenly and not, and the longest that the count takes whole."""
    sizes = [16385, 16896, 40000, 65536, 100, 9000] * len(KINDS) + [1 << 18]
    starts = _starts(sizes)
    keys = np.concatenate([_spread(KINDS[(i // 6 + i) % len(KINDS)], m, 90 + i)
                           for i, m in enumerate(sizes)])
    vals = [workloads.uniform_keys(len(keys), seed=81 + j) for j in range(max(vc, 0))]
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
    _check(oracle, keys, vals, vc, starts, g, fb, eb)
    assert any("_slots_b512_" in k for k in names) == (eb - fb > 16), names


def test_buckets_replayed(engine, oracle):
    """A captured plan over keys that go through buckets, then keys that take
    every pass, then both kinds, then buckets again."""
    import torch
    sizes = [20000, 30000, 50000, 65536, 100000, 17000]
    starts = _starts(sizes)
    n = int(starts[-1])
    vals = [np.arange(n, dtype=np.uint32)]
    g = GpuSort(np.zeros(n, dtype=np.uint32), vals, value_count=1)
    torch.cuda.synchronize()
    plan = engine.segmented_plan(g.data, starts)
    for r, kinds in enumerate([["uniform"], ["heavy"], ["uniform", "heavy"], ["narrow"],
                               ["uniform"]]):
        keys = np.concatenate([_spread(kinds[i % len(kinds)], m, 200 + 10 * r + i)
                               for i, m in enumerate(sizes)])
        g.by_ptr[g.data.keys[0]][:n].copy_(to_dev(keys, n))
        g.by_ptr[g.data.values[0][0]][:n].copy_(to_dev(vals[0], n))
        torch.cuda.synchronize()
        plan.execute(g.data)
        torch.cuda.synchronize()
        engine.check_device()
        _check(oracle, keys, vals, 1, starts, g, 0, 32)
    plan.close()


@pytest.mark.parametrize("vc,width", [(0, 32), (1, 32), (2, 24), (1, 16)])
def test_served_batch(engine, oracle, vc, width):
    """Requests of every class at once: on the server's one stream small ones
    and those between 8193 and 16384 keys join the buckets' launches (not with
    the two passes of 16 bits)."""
    import torch
    import mgpu_old_amd as mg
    from gpu_helpers import to_host
    sizes = [100, 1, 4096, 4097, 8192, 8193, 16384, 16385, 40000, 100000, 200000, 1 << 18]
    reqs, host = [], []
    for i, n in enumerate(sizes):
        keys = _spread(KINDS[i % len(KINDS)], n, 300 + i)
        vals = [workloads.uniform_keys(n, seed=400 + 10 * i + j) for j in range(vc)]
        tk, tv = to_dev(keys), [to_dev(v) for v in vals]
        r = mg.SortRequest()
        r.keys = tk.data_ptr()
        for j, t in enumerate(tv):
            r.values[j] = t.data_ptr()
        r.numElements, r.valueCount, r.firstBit, r.endBit = n, vc, 0, width
        reqs.append(r)
        host.append((keys, vals, tk, tv))
    torch.cuda.synchronize()
    with mg.Server(engine, 1 << 30, max_in_flight=2, max_elements=1 << 18) as srv:
        comps = srv.replay(reqs, np.zeros(len(reqs)))
    torch.cuda.synchronize()
    for i, (c, (keys, vals, tk, tv)) in enumerate(zip(comps, host)):
        assert c.status == 0, f"request {i} failed: {mg.status_string(c.status)}"
        rk, rv = oracle.stable_sort(keys, vals, first_bit=0, end_bit=width)
        assert np.array_equal(to_host(tk, keys.size), rk), f"request {i} keys differ"
        for j, t in enumerate(tv):
            assert np.array_equal(to_host(t, keys.size), rv[j]), f"request {i} values[{j}] differ"
