"""The workgroup sorts check the plan they are given (needs a gfx950 GPU).

Buckets and whole segments are planned by kernels from counts, or by the host;
one that is larger than a workgroup sorts, or reaches past its array, can only
come of a broken count.  The kernels are launched here with such plans by hand:
they sort nothing of it and report code 8.  The layouts of their arguments are
taken from kernel_args.h as it is, and members that are not set here are zero: a
layout written out a second time would, once the header goes on without it, give
the kernels pointers that are none."""
import ctypes
import os
import struct
import subprocess

import numpy as np
import pytest

import mgpu_old_amd as mg
from gpu_helpers import empty_dev, to_dev, to_host
from mgpu_old_amd import build
from test_gpu_layout import OBJECTS, _number_offset

pytestmark = pytest.mark.gpu

P = ctypes.c_void_p
MEMBERS = {
    "mgpuLocalArgs": ["keys_in", "keys_out", "n", "num_bits", "plan", "hist", "starts",
                      "num_passes", "last_width", "error_flag"],
    "mgpuMidPlan": ["buckets", "start", "bits"],
    "mgpuSegDesc": ["keys", "n", "route"],
    "mgpuSegSlotArgs": ["segs", "wide", "slots", "digit_start", "result_side", "num_bits",
                        "error_flag"],
}


@pytest.fixture(scope="module")
def layouts(tmp_path_factory):
    """Per structure: its size, and each member's offset and element size."""
    for name in OBJECTS:  # built from this header?
        data = open(os.path.join(mg.LIB_DIR, name), "rb").read()
        assert struct.unpack_from("<I", data, _number_offset(data))[0] == build.args_layout()
    src = tmp_path_factory.mktemp("layouts") / "layouts.cpp"
    lines = []
    for s, members in MEMBERS.items():
        lines.append(f'std::printf("{s} - %zu 0\\n", sizeof({s}));')
        lines += [f'std::printf("{s} {m} %zu %zu\\n", offsetof({s}, {m}), '
                  f"sizeof(std::remove_all_extents_t<decltype({s}::{m})>));" for m in members]
    src.write_text("#include <cstddef>\n#include <cstdio>\n#include <type_traits>\n"
                   '#include "kernel_args.h"\nint main() {\n' + "\n".join(lines) + "\n}\n")
    exe = str(src) + ".out"
    subprocess.run(["g++", "-std=c++17", "-I", build.CSRC, str(src), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    found = {s: {} for s in MEMBERS}
    for line in out.splitlines():
        s, m, at, size = line.split()
        found[s][m] = (int(at), int(size))
    return found


def _block(layouts, name, **members):
    """The structure's bytes: numbers, or a list for the first elements of an array."""
    lay = layouts[name]
    data = bytearray(lay["-"][0])
    for m, v in members.items():
        at, size = lay[m]
        for i, x in enumerate(v if isinstance(v, list) else [v]):
            struct.pack_into("<Q" if size == 8 else "<I", data, at + i * size, x)
    return data


def _launch(obj, name, grid, threads, args):
    import torch
    torch.cuda.synchronize()
    hip = ctypes.CDLL("libamdhip64.so")
    mod, fn = P(), P()
    assert hip.hipModuleLoad(ctypes.byref(mod), os.path.join(mg.LIB_DIR, obj).encode()) == 0
    assert hip.hipModuleGetFunction(ctypes.byref(fn), mod, name.encode()) == 0
    block = ctypes.create_string_buffer(bytes(args), len(args))
    params = (P * 1)(ctypes.cast(block, P))
    assert hip.hipModuleLaunchKernel(fn, grid, 1, 1, threads, 1, 1, 0, None, params, None) == 0
    torch.cuda.synchronize()
    assert hip.hipModuleUnload(mod) == 0


def _dev(data):
    return to_dev(np.frombuffer(bytes(data), dtype=np.uint32).copy())


# The first bucket's keys, of `n` in all.
@pytest.mark.parametrize("begin,size,n,code", [
    (0, 16384, 20_000, 0), (0, 16385, 20_000, 8), (19_000, 1001, 20_000, 8),
    (20_001, 5, 20_000, 8), (19_000, 1000, 20_000, 0)])
def test_bucket_of_an_array(layouts, begin, size, n, code):
    keys = np.random.default_rng(size).integers(0, 1 << 32, n, dtype=np.uint32)
    src, out, flag = to_dev(keys), to_dev(keys), to_dev(np.zeros(1, np.uint32))
    plan = _block(layouts, "mgpuMidPlan", buckets=1, start=[begin] + [begin + size] * 256,
                  bits=[32] * 256)
    dev_plan, scratch = _dev(plan), empty_dev(4096)
    a = _block(layouts, "mgpuLocalArgs", keys_in=src.data_ptr(), keys_out=out.data_ptr(), n=n,
               num_bits=32, plan=dev_plan.data_ptr(), hist=scratch.data_ptr(),
               starts=scratch.data_ptr(), num_passes=0, last_width=8, error_flag=flag.data_ptr())
    _launch("mgpusort_radix.hsaco", "mgpu_local_sort_k", 256, 1024, a)
    assert to_host(flag, 1)[0] == code
    want = keys.copy()
    if not code:
        want[begin:begin + size] = np.sort(keys[begin:begin + size])
    assert np.array_equal(to_host(out, n), want)


# A slot's workgroup: a whole segment (begin None) or a bucket of one.
@pytest.mark.parametrize("threads,most", [(512, 8192), (1024, 16384)])
@pytest.mark.parametrize("begin,past", [(None, 0), (None, 1), (0, 0), (0, 1), (1000, 0)])
def test_slots(layouts, threads, most, begin, past):
    n = most + past if begin is None else most + 500
    size = most + past
    code = 8 if past or begin == 1000 else 0
    keys = np.random.default_rng(n).integers(0, 1 << 32, n, dtype=np.uint32)
    sides = [to_dev(keys), to_dev(keys)]
    flag = to_dev(np.zeros(1, np.uint32))
    seg = _dev(_block(layouts, "mgpuSegDesc", n=n, route=1 << 31,
                      keys=[s.data_ptr() for s in sides]))
    starts = np.zeros(4 * 256, np.uint32)
    starts[256:260] = [begin or 0, size, 32, 0]
    dev_starts = to_dev(starts)
    slots = to_dev(np.array([0, 0xFFFFFFFF if begin is None else 0], np.uint32))
    side = 1 if begin is None else 0
    a = _block(layouts, "mgpuSegSlotArgs", segs=seg.data_ptr(), wide=seg.data_ptr(),
               slots=slots.data_ptr(), digit_start=dev_starts.data_ptr(), result_side=side,
               num_bits=32, error_flag=flag.data_ptr())
    _launch("mgpusort_seg.hsaco", f"mgpu_seg_slots_b{threads}_k", 1, threads, a)
    assert to_host(flag, 1)[0] == code
    want = keys.copy()
    if not code:
        at = begin or 0
        want[at:at + size] = np.sort(keys[at:at + size])
    assert np.array_equal(to_host(sides[side], n), want)
