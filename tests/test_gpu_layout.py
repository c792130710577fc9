"""An engine refuses code objects of other argument layouts than its library's
before it launches anything (needs a gfx950 GPU)."""
import ctypes
import os
import shutil

import pytest

import mgpu_old_amd as mg
from mgpu_old_amd import build

pytestmark = pytest.mark.gpu

OBJECTS = ["mgpusort_radix.hsaco", "mgpusort_seg.hsaco"]


def _create(path):
    h = ctypes.c_void_p()
    st = mg.lib().sortCreateEngine((str(path) + "/").encode(), ctypes.byref(h))
    if h.value:
        mg.lib().sortReleaseEngine(h)
    return st


@pytest.mark.parametrize("other", [None] + OBJECTS)
def test_code_object_of_another_layout(tmp_path, other):
    number = build.args_layout().to_bytes(4, "little")
    for name in OBJECTS:
        data = open(os.path.join(mg.LIB_DIR, name), "rb").read()
        assert number in data, f"{name} is not built from this kernel_args.h"
        if name == other:
            data = data.replace(number, (build.args_layout() ^ 2).to_bytes(4, "little"))
        (tmp_path / name).write_bytes(data)
    for name in ("mgpusort_seg_tuning.txt", "mgpusort_sort_tuning.txt"):
        shutil.copy(os.path.join(mg.LIB_DIR, name), tmp_path / name)
    want = mg.SortStatus.KERNEL_ERROR if other else mg.SortStatus.SUCCESS
    assert _create(tmp_path) == want
