"""Which way a mid-sized array is sorted (needs a gfx950 GPU).

The result is the same whatever the device decides, so the route is read off
the other side's buffer: a bucketed sort leaves the scatter into buckets on side
1, or (odd passes) the input on side 0, where the digit passes leave the output
of the last pass but one.  It is compared with the rule worked out here."""
import numpy as np
import pytest

import mgpu_old_amd as mg
from mgpu_old_amd import workloads
from gpu_helpers import GpuSort, make_engine, to_host

pytestmark = pytest.mark.gpu

MOST = 16384  # keys that a workgroup sorts


@pytest.fixture(scope="module")
def engine():
    eng = make_engine()
    yield eng
    eng.close()


def _digits(keys, shift, width):
    return (keys >> np.uint32(shift)) & np.uint32((1 << width) - 1)


def _route(keys, fb, eb):
    """(name, bucket of each key) of the rule."""
    n, widths = keys.size, mg.plan_passes(eb - fb)
    bins = _digits(keys, eb - 10, 10)
    count = np.bincount(bins, minlength=1024)
    top = count.reshape(256, 4).sum(axis=1)
    if top.max() <= MOST:
        return "top", bins >> 2
    if count.max() <= MOST:
        of_bin = (np.cumsum(count) - count) // max(1024, n // 256 + 1)
        if np.bincount(of_bin, weights=count).max() <= MOST:
            return "bins", of_bin[bins].astype(np.uint32)
    if top.max() < n:
        return "passes", None
    shifts = fb + np.cumsum([0] + widths)
    for p in range(len(widths) - 2, 0, -1):
        d = _digits(keys, int(shifts[p]), widths[p])
        most = np.bincount(d).max()
        if most <= MOST:
            return "digit", d
        if most < n:
            return "passes", None
    return "pieces", _digits(keys, fb, widths[0])


def _keys(kind, n):
    u = workloads.uniform_keys(n, seed=n)
    if kind == "even":
        return u
    if kind == "ramp":  # six times denser at the top than at the bottom
        x = u.astype(np.float64) / 2.0**32
        return (np.minimum((np.sqrt(1 + 35 * x) - 1) / 5, 1 - 2.0**-32) * 2.0**32).astype(np.uint32)
    if kind == "normal":
        return np.random.default_rng(n).standard_normal(n).astype(np.float32).view(np.uint32)
    if kind == "low":
        return workloads.and3_keys(n, seed=n)
    if kind == "narrow":
        return u >> np.uint32(9)
    if kind == "mid":  # one digit in the middle varies
        return (u & np.uint32(0xFF0000)) | np.uint32(0x12000034)
    if kind == "twelve":
        return u & np.uint32(0xFFF)
    if kind == "tiny":
        return u & np.uint32(0x7F)
    if kind == "high_tiny":  # the same in the lowest digit above bit 7
        return ((u & np.uint32(0x7F)) << np.uint32(7)) | np.uint32(0x80000055)
    return np.full(n, 0x89ABCDEF, dtype=np.uint32)


CASES = [("even", 16385, "top"), ("even", 1 << 19, "top"), ("even", 3 << 20, "top"),
         ("normal", 30_001, "top"), ("normal", 150_001, "bins"), ("normal", 400_001, "passes"),
         ("ramp", 2_500_001, "bins"), ("low", 200_001, "passes"), ("low", 1_400_001, "passes"),
         ("narrow", 150_001, "digit"), ("mid", 1_000_001, "digit"), ("twelve", 100_001, "digit"),
         ("twelve", 300_001, "passes"), ("tiny", 16385, "pieces"), ("tiny", 1 << 19, "pieces"),
         ("tiny", 3 << 20, "pieces"), ("equal", 20_001, "pieces"), ("equal", 600_001, "pieces")]


def _run(engine, oracle, kind, n, vc, fb, eb, expect):
    keys = _keys(kind, n)
    vals = [workloads.uniform_keys(n, seed=90 + j) for j in range(max(vc, 0))]
    key_type = mg.KEYS_FLOAT32 if kind == "normal" else None
    mapped = oracle.key_transform(keys, key_type, True) if key_type else keys
    name, bucket = _route(mapped, fb, eb)
    assert name == expect
    g = GpuSort(keys, vals, value_count=vc, first_bit=fb, end_bit=eb)
    g.run(engine, key_type=key_type)
    engine.check_device()
    rk, rv = oracle.stable_sort(mapped, vals, value_count=vc, first_bit=fb, end_bit=eb)
    assert np.array_equal(g.keys(), oracle.key_transform(rk, key_type, False) if key_type else rk)
    for o, r in zip(g.values(), rv):
        assert np.array_equal(o, r)
    widths = mg.plan_passes(eb - fb)
    other = to_host(g.by_ptr[g.data.keys[1]], n)
    if len(widths) % 2:
        assert g.data.parity == 1
        assert np.array_equal(other, keys) == (name != "passes")
        return
    if name == "passes":
        want, _ = oracle.stable_sort(mapped, [], value_count=0, first_bit=fb, end_bit=eb - widths[-1])
    else:
        want = mapped[np.argsort(bucket, kind="stable")]
    assert np.array_equal(other, want), name


@pytest.mark.parametrize("kind,n,expect", CASES)
@pytest.mark.parametrize("vc", [-1, 0, 1, 3])
def test_route(engine, oracle, kind, n, expect, vc):
    _run(engine, oracle, kind, n, vc, 0, 32, expect)


@pytest.mark.parametrize("kind,n,expect", [
    ("even", 50_001, "top"), ("low", 1_200_001, "passes"), ("high_tiny", 200_001, "pieces"),
    ("high_tiny", 1_200_001, "pieces"), ("equal", 100_001, "pieces")])
@pytest.mark.parametrize("vc", [-1, 0, 1, 3])
def test_route_of_three_digits(engine, oracle, kind, n, expect, vc):
    _run(engine, oracle, kind, n, vc, 7, 31, expect)
