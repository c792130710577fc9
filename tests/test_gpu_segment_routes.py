"""Which way a long segment of a batch is sorted (needs a gfx950 GPU): its result
is the same, so the route is read off side 1, which the one scatter into buckets
leaves in order of the digit it went by, and the digit passes in order of all
digits but the last.  It is compared with the rule worked out here.  Batches hold
segments of both kinds beside ones that a workgroup sorts whole."""
import numpy as np
import pytest

import mgpu_old_amd as mg
from mgpu_old_amd import workloads
from gpu_helpers import GpuSort, make_engine, to_host

pytestmark = pytest.mark.gpu

WHOLE, LONGEST, BUCKET = 16384, 1 << 18, 8192


@pytest.fixture(scope="module")
def engine():
    eng = make_engine()
    yield eng
    eng.close()


def _keys(kind, n, seed):
    u = workloads.uniform_keys(n, seed=seed)
    if kind == "even":
        return u
    if kind == "twothird":  # two thirds with one top digit
        m = workloads.uniform_keys(n, seed=seed + 1) % 3 > 0
        return np.where(m, (u & np.uint32(0xFFFFFF)) | np.uint32(0x41000000), u)
    if kind == "sorted":  # few top digits, some segments with one
        return np.sort(u >> np.uint32(seed % 12))
    if kind == "narrow":
        return u >> np.uint32(9)
    if kind == "tiny":
        return u & np.uint32(0x7F)
    return np.full(n, 0x12345678, dtype=np.uint32)


def _side1(keys, wide_keys, cus):
    """What side 1 holds after the sort, and whether buckets were used."""
    n = keys.size
    digit = [(keys >> np.uint32(8 * p)) & np.uint32(255) for p in range(4)]
    count = [np.bincount(d, minlength=256) for d in digit]
    cap = min(5632, max(4096, wide_keys // (2 * cus)))
    want = -(-n // cap)
    size = -(-n // want)
    picked = [p for p in range(4) if count[p].max() < n]
    if not picked:
        return keys, True
    p = picked[-1]
    ex = np.cumsum(count[p]) - count[p]
    fits = np.bincount(ex // size, weights=count[p]).max() <= BUCKET
    if fits:
        return keys[np.argsort(digit[p], kind="stable")], True
    return keys[np.argsort(keys & np.uint32(0xFFFFFF), kind="stable")], False


SIZES = [16385, 20_000, 40_000, 70_001, 131_072, LONGEST, 5000, 300, 12_000]


@pytest.mark.parametrize("kinds", [["even"], ["twothird"], ["sorted"], ["equal"], ["tiny"],
                                   ["even", "twothird"], ["narrow", "twothird", "equal", "sorted"]])
@pytest.mark.parametrize("vc", [-1, 0, 1, 3])
# (0: long ones only and many, so that whole segments are dealt to XCDs.)
@pytest.mark.parametrize("repeat", [1, 4, 12, 0])
def test_routes(engine, oracle, kinds, vc, repeat):
    sizes = SIZES * repeat if repeat > 1 else SIZES[3:7] if repeat else SIZES[2:6] * 20
    starts = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    n = int(starts[-1])
    parts = [_keys(kinds[i % len(kinds)], s, seed=i) for i, s in enumerate(sizes)]
    keys = np.concatenate(parts)
    vals = [workloads.uniform_keys(n, seed=70 + j) for j in range(max(vc, 0))]
    g = GpuSort(keys, vals, value_count=vc)
    plan = engine.segmented_plan(g.data, starts)
    engine.enable_timing(True)  # (the plan's launches one by one, by name)
    engine.read_timing()
    plan.execute(g.data)
    engine.check_device()
    names = set(engine.read_timing())
    engine.enable_timing(False)
    if engine.info()["xcdSegments"] > 1:
        assert any("_xr_" in k for k in names) == (repeat == 0), names
    side1 = to_host(g.by_ptr[g.data.keys[1]], n)
    out, outs = g.keys(), g.values()
    wide = sum(s for s in sizes if s > WHOLE)
    assert wide >= 1 << 18
    routes = set()
    for i, s in enumerate(sizes):
        a, b = int(starts[i]), int(starts[i + 1])
        rk, rv = oracle.stable_sort(parts[i], [v[a:b] for v in vals], value_count=vc)
        assert np.array_equal(out[a:b], rk)
        for o, r in zip(outs, rv):
            assert np.array_equal(o[a:b], r)
        if s > WHOLE:
            want, buckets = _side1(parts[i], wide, engine.info()["numCUs"])
            assert np.array_equal(side1[a:b], want), (i, s, kinds[i % len(kinds)], buckets)
            routes.add(buckets)
    if kinds in (["even"], ["equal"]):
        assert routes == {True}
    if kinds == ["even", "twothird"]:
        assert routes == {True, False}
    plan.close()
