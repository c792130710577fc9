"""Arrays that one workgroup sorts in one launch (mgpu_local_sort_*): bit-exact
against the oracle at the edges of the keys-per-thread steps and of the range,
for every value mode, bit range and key type, on keys that take the ranking
with one add per key and the one for slots of equal digits."""
import numpy as np
import pytest

import mgpu_old_amd as mg
from mgpu_old_amd import workloads
from gpu_helpers import GpuSort, make_engine

pytestmark = pytest.mark.gpu

MAX = 16384


@pytest.fixture(scope="module")
def engine():
    eng = make_engine()
    yield eng
    eng.close()


def _keys(kind, n):
    if kind == "equal":
        return np.full(n, 0x5A5A5A5A, dtype=np.uint32)
    if kind == "sorted":
        return np.sort(workloads.uniform_keys(n, seed=n + 1))
    if kind == "low":
        return workloads.and3_keys(n, seed=n + 2)
    return workloads.uniform_keys(n, seed=n)


@pytest.mark.parametrize("n", [1, 64, 1023, 1024, 1025, 2049, 4095, 4097, 8191, 8193, 12287, 12289,
                               MAX - 1, MAX, MAX + 1])
@pytest.mark.parametrize("vc", [-1, 0, 1, 2, 6])
@pytest.mark.parametrize("kind", ["uniform", "equal", "sorted", "low"])
def test_one_launch_sort(engine, oracle, n, vc, kind):
    keys = _keys(kind, n)
    vals = [workloads.uniform_keys(n, seed=40 + j) for j in range(max(vc, 0))]
    for fb, eb in [(0, 32), (0, 24), (7, 25), (31, 32)]:
        g = GpuSort(keys, vals, value_count=vc, first_bit=fb, end_bit=eb)
        engine.enable_timing(True)
        engine.read_timing()
        g.run(engine)
        names = set(engine.read_timing())
        engine.enable_timing(False)
        assert (len(names) == 1) == (n <= MAX), names
        rk, rv = oracle.stable_sort(keys, vals, value_count=vc, first_bit=fb, end_bit=eb)
        assert np.array_equal(g.keys(), rk)
        for o, r in zip(g.values(), rv):
            assert np.array_equal(o, r)
        assert g.data.parity == len(mg.plan_passes(eb - fb)) % 2


@pytest.mark.parametrize("key_type", [mg.KEYS_INT32, mg.KEYS_FLOAT32])
@pytest.mark.parametrize("n", [1025, MAX])
def test_one_launch_sort_of_typed_keys(engine, oracle, key_type, n):
    keys = workloads.uniform_keys(n, seed=7)  # every bit pattern: NaNs and zeros of both signs too
    keys[:4] = [0x80000000, 0, 0x7FC00000, 0xFFC00000]
    mapped = oracle.key_transform(keys, key_type, True)
    for vc in (-1, 2):
        vals = [workloads.uniform_keys(n, seed=50 + j) for j in range(max(vc, 0))]
        g = GpuSort(keys, vals, value_count=vc).run(engine, key_type=key_type)
        rk, rv = oracle.stable_sort(mapped, vals, value_count=vc)
        assert np.array_equal(g.keys(), oracle.key_transform(rk, key_type, False))
        for o, r in zip(g.values(), rv):
            assert np.array_equal(o, r)
