"""sortArrayEx refuses what the caller's split refuses (needs a gfx950 GPU):
with generated indices and several passes asked for, values1[0] has to be
given, however few passes the engine takes."""
import ctypes

import numpy as np
import pytest

import mgpu_old_amd as mg
from mgpu_old_amd import workloads
from gpu_helpers import GpuSort, make_engine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    eng = make_engine()
    yield eng
    eng.close()


# (bits, bits a pass): one pass; three of them, which one could do; two.
@pytest.mark.parametrize("bits,per_pass,refused", [(6, 6, False), (8, 3, True), (7, 3, True),
                                                   (8, 4, True)])
@pytest.mark.parametrize("n", [0, 1000, 100_000])
def test_index_mode_without_values_0(engine, oracle, bits, per_pass, refused, n):
    import torch
    keys = workloads.uniform_keys(n, seed=n + bits)
    g = GpuSort(keys, value_count=-1, end_bit=bits)
    missing = g.data.values[0][0]
    g.data.values[0][0] = 0
    torch.cuda.synchronize()
    st = mg.lib().sortArrayEx(engine.handle, ctypes.byref(g.data), 256, 8, per_pass, False)
    torch.cuda.synchronize()
    if refused and n:
        assert st == mg.SortStatus.INVALID_VALUE
        assert g.data.parity == 0 and g.data.keys[0] == g.start_keys
        return
    assert st == mg.SortStatus.SUCCESS
    if n:
        rk, (ri,) = oracle.stable_sort(keys, value_count=-1, end_bit=bits)
        assert g.data.parity == 1
        assert np.array_equal(g.keys(), rk) and np.array_equal(g.values()[0], ri)
        assert g.data.values[0][1] == 0 and missing
