"""Captured sorts whose route is decided on the device, replayed on keys that take
another one each time, with eager sorts on the same engine in between; and typed
keys through the launch that sorts buckets or makes a pass (needs a gfx950 GPU)."""
import numpy as np
import pytest

import mgpu_old_amd as mg
from mgpu_old_amd import workloads
from gpu_helpers import GpuSort, make_engine, to_dev

pytestmark = pytest.mark.gpu


def _keys(kind, n, seed):
    u = workloads.uniform_keys(n, seed=seed)
    if kind == "low":
        return workloads.and3_keys(n, seed=seed)
    if kind == "tiny":
        return u & np.uint32(0x7F)
    if kind == "narrow":
        return u >> np.uint32(9)
    if kind == "twothird":
        m = workloads.uniform_keys(n, seed=seed + 1) % 3 > 0
        return np.where(m, (u & np.uint32(0xFFFFFF)) | np.uint32(0x41000000), u)
    return u


def _refill(g, keys, vals):
    n = keys.size
    g.by_ptr[g.data.keys[0]][:n].copy_(to_dev(keys))
    for j, v in enumerate(vals):
        g.by_ptr[g.data.values[j][0]][:n].copy_(to_dev(v))


# Above 2^20 keys: the pass after the scatter and the buckets' sort in one launch.
@pytest.mark.parametrize("vc", [0, 1, 3])
def test_captured_array(oracle, vc):
    import torch
    n = 1_300_001
    eng = make_engine()
    stream = torch.cuda.Stream()
    try:
        eng.set_stream(stream.cuda_stream)
        vals = [workloads.uniform_keys(n, seed=5 + j) for j in range(vc)]
        g = GpuSort(np.zeros(n, dtype=np.uint32), vals)
        torch.cuda.synchronize()
        eng.sort_array(g.data)  # scratch of this size
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            eng.sort_array(g.data)
        for r, kind in enumerate(["even", "low", "even", "tiny", "low", "narrow"]):
            other = GpuSort(_keys("low", 700_001, r)).run(eng)
            assert np.array_equal(other.keys(), np.sort(_keys("low", 700_001, r)))
            keys = _keys(kind, n, 20 + r)
            _refill(g, keys, vals)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            eng.check_device()
            rk, rv = oracle.stable_sort(keys, vals)
            assert np.array_equal(g.keys(), rk), kind
            for o, v in zip(g.values(), rv):
                assert np.array_equal(o, v), kind
    finally:
        eng.close()


# Long segments dealt to XCDs, and shorter ones beside small and whole ones.
@pytest.mark.parametrize("sizes", [[40_000, 70_001, 131_072, 1 << 18] * 20,
                                   [300, 5000, 9000, 20_000, 40_000, 100_000] * 6])
@pytest.mark.parametrize("vc", [0, 1, 2])
def test_plan(oracle, sizes, vc):
    import torch
    starts = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    n = int(starts[-1])
    eng = make_engine()
    vals = [workloads.uniform_keys(n, seed=7 + j) for j in range(vc)]
    g = GpuSort(np.zeros(n, dtype=np.uint32), vals)
    torch.cuda.synchronize()
    plan = eng.segmented_plan(g.data, starts)
    for r, kinds in enumerate([["even"], ["twothird"], ["even", "twothird", "tiny"], ["low"],
                               ["even"]]):
        parts = [_keys(kinds[i % len(kinds)], s, 100 * r + i) for i, s in enumerate(sizes)]
        _refill(g, np.concatenate(parts), vals)
        torch.cuda.synchronize()
        plan.execute(g.data)
        torch.cuda.synchronize()
        eng.check_device()
        out, outs = g.keys(), g.values()
        for i in range(len(sizes)):
            a, b = int(starts[i]), int(starts[i + 1])
            rk, rv = oracle.stable_sort(parts[i], [v[a:b] for v in vals])
            assert np.array_equal(out[a:b], rk), (r, i)
            for o, v in zip(outs, rv):
                assert np.array_equal(o[a:b], v), (r, i)
    plan.close()
    eng.close()


@pytest.mark.parametrize("key_type", [mg.KEYS_INT32, mg.KEYS_FLOAT32])
@pytest.mark.parametrize("kind", ["even", "low", "tiny"])
@pytest.mark.parametrize("n", [600_001, 1_300_001])
def test_typed_keys(oracle, key_type, kind, n):
    eng = make_engine()
    keys = _keys(kind, n, 3)
    mapped = oracle.key_transform(keys, key_type, True)
    for vc in (-1, 0, 1, 2):
        vals = [workloads.uniform_keys(n, seed=80 + j) for j in range(max(vc, 0))]
        g = GpuSort(keys, vals, value_count=vc).run(eng, key_type=key_type)
        eng.check_device()
        rk, rv = oracle.stable_sort(mapped, vals, value_count=vc)
        assert np.array_equal(g.keys(), oracle.key_transform(rk, key_type, False))
        for o, r in zip(g.values(), rv):
            assert np.array_equal(o, r)
    eng.close()
