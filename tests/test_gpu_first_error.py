"""The error word keeps the first code of a failure (needs a gfx950 GPU).

Every lookback is made to give up (MGPUSORT_SPIN_LIMIT=0), so the first pass
reports code 1 and leaves parts of its output unwritten.  Those hold all ones
here, far more keys of the top digit than were counted, so the passes after it
find scatter offsets out of range (code 4, dropped by the stores' range check):
a consequence, which must not take the place of the cause.
"""
import numpy as np
import pytest

import mgpu_old_amd as mg
from mgpu_old_amd import workloads
from gpu_helpers import GpuSort, make_engine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def failing():
    eng = make_engine({"MGPUSORT_SPIN_LIMIT": "0"})
    yield eng
    eng.close()


def _ones_on_side_1(g):
    import torch
    g.by_ptr[g.data.keys[1]].fill_(-1)
    torch.cuda.synchronize()


def _first_code(engine):
    code = engine.info()["deviceError"]
    assert mg.lib().sortCheckDevice(engine.handle) == mg.SortStatus.KERNEL_ERROR
    assert mg.lib().sortCheckDevice(engine.handle) == mg.SortStatus.SUCCESS
    return code


# Passes after a bucketed sort's scatter in one launch, and a launch each; one
# lookback chain; a chain per XCD.
@pytest.mark.parametrize("n", [300_001, (1 << 20) + 1, (1 << 22) + 1, 1 << 24])
@pytest.mark.parametrize("vc", [0, 1])
def test_array(failing, n, vc):
    keys = workloads.and3_keys(n, seed=n)
    g = GpuSort(keys, [np.arange(n, dtype=np.uint32)][:vc])
    _ones_on_side_1(g)
    g.run(failing)
    assert _first_code(failing) == 1


@pytest.mark.parametrize("size", [200_000, 300_000])
def test_segments(failing, size):
    starts = np.arange(5, dtype=np.int64) * size
    keys = workloads.and3_keys(int(starts[-1]), seed=size)
    g = GpuSort(keys)
    _ones_on_side_1(g)
    plan = failing.segmented_plan(g.data, starts)
    plan.execute(g.data)
    assert _first_code(failing) == 1
    plan.close()
