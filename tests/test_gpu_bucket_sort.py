"""Mid-sized arrays, sorted in buckets (mgpu_mid_count, the _m_ scatter and a
workgroup's sort per bucket, or the digit passes where a bucket does not fit):
bit-exact against the oracle at the edges of the range and of its launch
shapes, for keys that take each way of forming buckets and for keys that take
none."""
import numpy as np
import pytest

import mgpu_old_amd as mg
from mgpu_old_amd import workloads
from gpu_helpers import GpuSort, make_engine, to_dev

pytestmark = pytest.mark.gpu

FIRST, LAST = 16385, 3 << 20


@pytest.fixture(scope="module")
def engine():
    eng = make_engine()
    yield eng
    eng.close()


def _keys(kind, n):
    u = workloads.uniform_keys(n, seed=n)
    if kind == "even":  # 4 bins a bucket
        return u
    if kind == "skewed":  # bins grouped by their counts: squares of even words
        f = u.astype(np.float64) / 2.0**32
        return np.minimum(f * f * 2.0**32, 2.0**32 - 1).astype(np.uint32)
    if kind == "narrow":  # constant top digits: buckets of a lower digit
        return u >> np.uint32(9)
    if kind == "small":  # every key below 2^12: no digit spreads them enough
        return u & np.uint32(0xFFF)
    if kind == "low":
        return workloads.and3_keys(n, seed=n + 1)
    if kind == "one_bin":  # half of the keys in one bin
        return np.where(u & np.uint32(1), u, u & np.uint32(0x3FFFFF))
    return np.full(n, 0xFFFFFFFF, dtype=np.uint32)


def _check(oracle, keys, g, vals, vc, fb=0, eb=32):
    rk, rv = oracle.stable_sort(keys, vals, value_count=vc, first_bit=fb, end_bit=eb)
    assert np.array_equal(g.keys(), rk)
    for o, r in zip(g.values(), rv):
        assert np.array_equal(o, r)


@pytest.mark.parametrize("kind", ["even", "skewed", "narrow", "small", "low", "one_bin", "equal"])
@pytest.mark.parametrize("n", [FIRST, 65536, 150_001, (1 << 19), (1 << 19) + 1, (1 << 20) + 1])
@pytest.mark.parametrize("vc", [-1, 0, 1, 2])
def test_bucket_sort(engine, oracle, kind, n, vc):
    keys = _keys(kind, n)
    vals = [workloads.uniform_keys(n, seed=60 + j) for j in range(max(vc, 0))]
    g = GpuSort(keys, vals, value_count=vc)
    engine.enable_timing(True)
    engine.read_timing()
    g.run(engine)
    names = set(engine.read_timing())
    engine.enable_timing(False)
    engine.check_device()
    assert "mgpu_mid_count" in names
    assert any("_f_" in k for k in names) == (n <= 1 << 19), names
    _check(oracle, keys, g, vals, vc)
    assert g.data.parity == 0


@pytest.mark.parametrize("kind", ["even", "skewed", "low"])
@pytest.mark.parametrize("n", [LAST, LAST + 1])
def test_largest(engine, oracle, kind, n):
    keys = _keys(kind, n)
    vals = [np.arange(n, dtype=np.uint32)]
    engine.enable_timing(True)
    engine.read_timing()
    g = GpuSort(keys, vals).run(engine)
    names = set(engine.read_timing())
    engine.enable_timing(False)
    engine.check_device()
    assert ("mgpu_mid_count" in names) == (n <= LAST), names
    _check(oracle, keys, g, vals, 1)


@pytest.mark.parametrize("fb,eb", [(0, 17), (7, 25), (15, 32), (8, 32), (3, 27), (2, 32)])
@pytest.mark.parametrize("kind", ["even", "low", "narrow"])
@pytest.mark.parametrize("n", [20_001, 700_001])
def test_bit_ranges(engine, oracle, fb, eb, kind, n):
    keys = _keys(kind, n)
    vals = [workloads.uniform_keys(n, seed=70 + j) for j in range(3)]
    for vc in (-1, 3):
        v = vals if vc == 3 else []
        g = GpuSort(keys, v, value_count=vc, first_bit=fb, end_bit=eb).run(engine)
        _check(oracle, keys, g, v, vc, fb, eb)
        assert g.data.parity == len(mg.plan_passes(eb - fb)) % 2


@pytest.mark.parametrize("key_type", [mg.KEYS_INT32, mg.KEYS_FLOAT32])
@pytest.mark.parametrize("n", [30_001, 150_001, 900_001])
def test_typed_keys(engine, oracle, key_type, n):
    rng = np.random.default_rng(n)
    if key_type == mg.KEYS_FLOAT32:
        keys = rng.standard_normal(n).astype(np.float32)
        keys[:5] = [np.inf, -np.inf, np.nan, 0.0, -0.0]
        keys = keys.view(np.uint32)
    else:
        keys = rng.integers(-1000, 1000, n, dtype=np.int32).view(np.uint32)
    mapped = oracle.key_transform(keys, key_type, True)
    for vc in (0, 1):
        vals = [workloads.uniform_keys(n, seed=80)][:vc]
        g = GpuSort(keys, vals, value_count=vc).run(engine, key_type=key_type)
        rk, rv = oracle.stable_sort(mapped, vals, value_count=vc)
        assert np.array_equal(g.keys(), oracle.key_transform(rk, key_type, False))
        for o, r in zip(g.values(), rv):
            assert np.array_equal(o, r)


def test_captured(oracle):
    """A captured bucket sort replayed on new inputs, buckets used or not, with
    eager sorts on the engine in between."""
    import torch
    n = 100_001
    eng = make_engine()
    stream = torch.cuda.Stream()
    try:
        eng.set_stream(stream.cuda_stream)
        g = GpuSort(np.zeros(n, dtype=np.uint32), [np.arange(n, dtype=np.uint32)])
        torch.cuda.synchronize()
        eng.sort_array(g.data)  # scratch of this size
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            eng.sort_array(g.data)
        vals = np.arange(n, dtype=np.uint32)
        for kind in ("even", "low", "even", "equal", "skewed"):
            keys = _keys(kind, n)
            other = GpuSort(_keys("low", 50_001)).run(eng)
            assert np.array_equal(other.keys(), np.sort(_keys("low", 50_001)))
            g.by_ptr[g.data.keys[0]][:n].copy_(to_dev(keys))
            g.by_ptr[g.data.values[0][0]][:n].copy_(to_dev(vals))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            eng.check_device()
            _check(oracle, keys, g, [vals], 1)
    finally:
        eng.close()


@pytest.mark.parametrize("fb,eb", [(0, 32), (0, 31), (5, 30), (0, 24), (4, 20), (0, 13), (0, 7)])
@pytest.mark.parametrize("n", [3000, 40_001, 3 * (1 << 20) + 5])
def test_ex_runs_fewer_passes(engine, oracle, fb, eb, n):
    """sortArrayEx with every digit width: the order, the parity and the side of
    the result are those of the caller's passes, however many run."""
    if n > 1 << 20 and (fb, eb) not in ((0, 32), (0, 24)):
        return
    keys = _keys("even", n)
    vals = [np.arange(n, dtype=np.uint32)]
    rk, (rv,) = oracle.stable_sort(keys, vals, first_bit=fb, end_bit=eb)
    for bit_pass in (1, 2, 3, 4, 5, 6):
        g = GpuSort(keys, vals, first_bit=fb, end_bit=eb)
        g.run(engine, ex=(256, 8, bit_pass, False))
        engine.check_device()
        assert np.array_equal(g.keys(), rk) and np.array_equal(g.values()[0], rv)
        passes = -(-(eb - fb) // min(bit_pass, eb - fb))
        assert g.data.parity == passes % 2
        assert g.data.keys[g.data.parity] == g.start_keys
