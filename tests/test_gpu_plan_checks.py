"""The workgroup sorts check the plan they are given (needs a gfx950 GPU).

Buckets and whole segments are planned by kernels from counts, or by the host;
one that is larger than a workgroup sorts, or reaches past its array, can only
come of a broken count.  The kernels are launched here with such plans by hand:
they sort nothing of it and report code 8."""
import ctypes
import os

import numpy as np
import pytest

import mgpu_old_amd as mg
from gpu_helpers import empty_dev, to_dev, to_host

pytestmark = pytest.mark.gpu

P, U = ctypes.c_void_p, ctypes.c_uint32


class LocalArgs(ctypes.Structure):  # mgpuLocalArgs
    _fields_ = [("keys_in", P), ("keys_out", P), ("vals_in", P * 6), ("vals_out", P * 6),
                ("n", U), ("first_bit", U), ("num_bits", U), ("vals_mode", U), ("num_values", U),
                ("in_lo", U), ("in_hi", U), ("out_lo", U), ("out_hi", U), ("pad", U),
                ("plan", P), ("hist", P), ("starts", P), ("num_passes", U), ("last_width", U),
                ("error_flag", P)]


class Plan(ctypes.Structure):  # mgpuMidPlan
    _fields_ = [("buckets", U), ("pad", U * 3), ("start", U * 257), ("base", U * 256),
                ("bits", U * 256), ("pad2", U * 3)]


class Desc(ctypes.Structure):  # mgpuSegDesc
    _fields_ = [("keys", P * 2), ("vals", (P * 2) * 6), ("n", U), ("route", U)]


class SlotArgs(ctypes.Structure):  # mgpuSegSlotArgs
    _fields_ = [("segs", P), ("wide", P), ("slots", P), ("digit_start", P),
                ("num_values", U), ("index_mode", U), ("result_side", U), ("first_bit", U),
                ("num_bits", U), ("pad", U), ("error_flag", P)]


def _launch(obj, name, grid, threads, args):
    import torch
    torch.cuda.synchronize()
    hip = ctypes.CDLL("libamdhip64.so")
    mod, fn = P(), P()
    assert hip.hipModuleLoad(ctypes.byref(mod), os.path.join(mg.LIB_DIR, obj).encode()) == 0
    assert hip.hipModuleGetFunction(ctypes.byref(fn), mod, name.encode()) == 0
    params = (P * 1)(ctypes.cast(ctypes.pointer(args), P))
    assert hip.hipModuleLaunchKernel(fn, grid, 1, 1, threads, 1, 1, 0, None, params, None) == 0
    torch.cuda.synchronize()
    assert hip.hipModuleUnload(mod) == 0


def _dev(struct):
    return to_dev(np.frombuffer(bytes(struct), dtype=np.uint32).copy())


# The first bucket's keys, of `n` in all.
@pytest.mark.parametrize("begin,size,n,code", [
    (0, 16384, 20_000, 0), (0, 16385, 20_000, 8), (19_000, 1001, 20_000, 8),
    (20_001, 5, 20_000, 8), (19_000, 1000, 20_000, 0)])
def test_bucket_of_an_array(begin, size, n, code):
    keys = np.random.default_rng(size).integers(0, 1 << 32, n, dtype=np.uint32)
    src, out, flag = to_dev(keys), to_dev(keys), to_dev(np.zeros(1, np.uint32))
    plan = Plan(buckets=1)
    plan.start[0] = begin
    for b in range(1, 257):
        plan.start[b] = begin + size
    for b in range(256):
        plan.bits[b] = 32
    dev_plan, scratch = _dev(plan), empty_dev(4096)
    a = LocalArgs(keys_in=src.data_ptr(), keys_out=out.data_ptr(), n=n, num_bits=32,
                  plan=dev_plan.data_ptr(), hist=scratch.data_ptr(), starts=scratch.data_ptr(),
                  num_passes=0, last_width=8, error_flag=flag.data_ptr())
    _launch("mgpusort_radix.hsaco", "mgpu_local_sort_k", 256, 1024, a)
    assert to_host(flag, 1)[0] == code
    want = keys.copy()
    if not code:
        want[begin:begin + size] = np.sort(keys[begin:begin + size])
    assert np.array_equal(to_host(out, n), want)


# A slot's workgroup: a whole segment (begin None) or a bucket of one.
@pytest.mark.parametrize("threads,most", [(512, 8192), (1024, 16384)])
@pytest.mark.parametrize("begin,past", [(None, 0), (None, 1), (0, 0), (0, 1), (1000, 0)])
def test_slots(threads, most, begin, past):
    n = most + past if begin is None else most + 500
    size = most + past
    code = 8 if past or begin == 1000 else 0
    keys = np.random.default_rng(n).integers(0, 1 << 32, n, dtype=np.uint32)
    sides = [to_dev(keys), to_dev(keys)]
    flag = to_dev(np.zeros(1, np.uint32))
    d = Desc(n=n, route=1 << 31)
    for s in (0, 1):
        d.keys[s] = sides[s].data_ptr()
    seg = _dev(d)
    starts = np.zeros(4 * 256, np.uint32)
    starts[256:260] = [begin or 0, size, 32, 0]
    dev_starts = to_dev(starts)
    slots = to_dev(np.array([0, 0xFFFFFFFF if begin is None else 0], np.uint32))
    a = SlotArgs(segs=seg.data_ptr(), wide=seg.data_ptr(), slots=slots.data_ptr(),
                 digit_start=dev_starts.data_ptr(),
                 result_side=1 if begin is None else 0, num_bits=32, error_flag=flag.data_ptr())
    _launch("mgpusort_seg.hsaco", f"mgpu_seg_slots_b{threads}_k", 1, threads, a)
    assert to_host(flag, 1)[0] == code
    want = keys.copy()
    if not code:
        at = begin or 0
        want[at:at + size] = np.sort(keys[at:at + size])
    assert np.array_equal(to_host(sides[a.result_side], n), want)
