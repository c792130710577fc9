"""An engine refuses code objects of other argument layouts than its library's
before it launches anything (needs a gfx950 GPU)."""
import ctypes
import os
import shutil
import struct

import pytest

import mgpu_old_amd as mg

pytestmark = pytest.mark.gpu

OBJECTS = ["mgpusort_radix.hsaco", "mgpusort_seg.hsaco"]


def _create(path):
    h = ctypes.c_void_p()
    st = mg.lib().sortCreateEngine((str(path) + "/").encode(), ctypes.byref(h))
    if h.value:
        mg.lib().sortReleaseEngine(h)
    return st


def _number_offset(data):
    """File offset of the layout number in a code object (ELF64)."""
    shoff, = struct.unpack_from("<Q", data, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", data, 0x3A)
    sections = [struct.unpack_from("<IIQQQQIIQQ", data, shoff + i * shentsize) for i in range(shnum)]
    for sec in sections:
        if sec[1] not in (2, 11):  # SHT_SYMTAB, SHT_DYNSYM
            continue
        names = sections[sec[6]][4]
        for at in range(sec[4], sec[4] + sec[5], sec[9]):
            name, _, _, shndx, value, size = struct.unpack_from("<IBBHQQ", data, at)
            end = data.index(b"\0", names + name)
            if data[names + name:end] == b"mgpu_args_layout":
                assert size == 4
                return value - sections[shndx][3] + sections[shndx][4]
    raise AssertionError("no layout number")


@pytest.mark.parametrize("other", [None] + OBJECTS)
def test_code_object_of_another_layout(tmp_path, other):
    for name in OBJECTS:
        data = bytearray(open(os.path.join(mg.LIB_DIR, name), "rb").read())
        if name == other:
            data[_number_offset(data)] ^= 2
        (tmp_path / name).write_bytes(data)
    for name in ("mgpusort_seg_tuning.txt", "mgpusort_sort_tuning.txt"):
        shutil.copy(os.path.join(mg.LIB_DIR, name), tmp_path / name)
    want = mg.SortStatus.KERNEL_ERROR if other else mg.SortStatus.SUCCESS
    assert _create(tmp_path) == want
