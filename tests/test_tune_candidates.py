"""What the autotuners time (mgpu_old_amd/tune_sort.py, tune_segsort.py)."""
import pytest

from mgpu_old_amd import tune_segsort, tune_sort


def test_every_choice_is_a_candidate():
    assert sorted(tune_sort.CANDIDATES) == sorted(
        (t, c) for t in ("small", "large") for c in ("one", "xcd"))
    rows = [r.split() for r in tune_sort.candidate_table("small", "xcd").splitlines()]
    assert [r[0] for r in rows] == ["31"] * len(tune_sort.CLASSES)
    assert [r[1] for r in rows] == list(tune_sort.CLASSES)
    assert all(r[2:] == ["small", "xcd"] for r in rows)


def test_kept_keys_are_searched():
    kept = {line.split()[-1] for line in tune_segsort.wide_lines()}
    assert {"0", "16384"} <= kept and len(kept) > 2


@pytest.mark.gpu
@pytest.mark.parametrize("tile,block", [("small", "_b512_"), ("large", "_b1024_")])
def test_candidate_takes_the_route_of_its_size(tmp_path, tile, block):
    """A mid-sized array of a candidate goes through buckets, as it does with
    the table that the tuner writes."""
    import torch
    import mgpu_old_amd as mg
    from mgpu_old_amd import workloads
    n = 1 << 18
    eng = tune_sort.make_engine(mg, torch, str(tmp_path), tune_sort.candidate_table(tile, "one"))
    src = workloads.uniform_keys_torch(n, 5, "cuda", torch=torch)
    eng.enable_timing(True)
    tune_sort.time_sort(torch, mg, eng, n, 1, src, 1)
    names = set(eng.read_timing())
    eng.close()
    assert "mgpu_mid_count" in names
    scatter = {k for k in names if k.startswith("mgpu_rank_scatter")}
    assert scatter and all(block in k for k in scatter), names
