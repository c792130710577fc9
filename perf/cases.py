"""The sort's working set for performance measurements.

Each case is one call pattern of the library: `prepare` makes what a program
holds before the call (inputs, buffers, an engine, a captured plan or a sort
server), `run` is one pass through the public entry points, `work` the bytes
the call cannot do without, `exact` the same result from torch alone.

A sort works in place, so a pass first puts its input into the sort's buffers
with one elementwise kernel, as the producer of the keys would in a program
that sorts new data every time; keys and values lie in one allocation, so it
is one launch.
"""
import math

import numpy as np
import torch

import mgpu_old_amd as mg

_DEV = "cuda"
_TYPES = {"uint32": mg.KEYS_UINT32, "int32": mg.KEYS_INT32, "float32": mg.KEYS_FLOAT32}


def _sort(name, n, values=0, first=0, end=32, keys="uniform", type="uint32", call="array"):
    """One array: n keys with `values` value arrays (-1: generated indices)."""
    return {"name": name, "kind": call, "n": n, "values": values, "first": first, "end": end,
            "keys": keys, "type": type}


def _segments(name, kind, count, lo, hi, values):
    """count arrays whose sizes are log-uniform in [lo, hi]."""
    return {"name": name, "kind": kind, "count": count, "lo": lo, "hi": hi, "values": values,
            "first": 0, "end": 32, "keys": "uniform", "type": "uint32"}


def listed():
    return [
        # A short list sorted on the way to something else: latency only.
        _sort("pair_1k", 1000, 1),
        # Argsort of a small table by a 24-bit field, ragged size.
        _sort("argsort_20k_24bit", 20001, -1, 0, 24),
        # Depth or score order: float keys with an id.
        _sort("float_pair_150k", 150000, 1, type="float32"),
        # The caller fixes the digit width (the reference's smallsort size).
        _sort("ex6_pair_500k", 500000, 1, call="ex"),
        # The benchmark's keys-only workload.
        _sort("keys_1m", 1 << 20),
        # Records of three payload words ordered by a field inside the key.
        _sort("triple_3m_field", 3000001, 3, 7, 25),
        # The benchmark's mid-size and headline key + value workloads.
        _sort("pair_32m", 1 << 25, 1),
        _sort("pair_256m", 1 << 28, 1),
        # Low-entropy 24-bit keys with generated indices, large.
        _sort("index_128m_low_24bit", 1 << 27, -1, 0, 24, "low"),
        # The benchmark's ragged batch, replayed from a captured plan.
        _segments("plan_4096_ragged", "plan", 4096, 1, 1 << 16, 1),
        # Many short lists (rows of a sparse matrix), replayed.
        _segments("plan_60k_short", "plan", 60000, 1, 512, 0),
        # A burst of independent requests through the sort service.
        _segments("served_96", "serve", 96, 1 << 10, 1 << 18, 1),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["array"] * 6 + ["ex", "plan", "plan", "serve"])
    if kind in ("plan", "serve"):
        values = rng.choice([-1, 0, 1, 1, 2]) if kind == "plan" else rng.choice([0, 1, 1])
        hi = log(16, 1 << 18)
        lo = max(1, log(1, hi))
        # About 2^20 to 2^24 keys for a plan, a few million for a burst.
        mean = (hi - lo) / max(1e-9, math.log(hi / lo)) if hi > lo else hi
        count = int(log(1 << 20, 1 << 24) / mean) if kind == "plan" else int(log(1 << 18, 1 << 22) / mean)
        count = max(8, min(100000 if kind == "plan" else 400, count))
        case = _segments("", kind, count, lo, hi, values)
    else:
        n = log(300, 1 << 27) if kind == "array" else log(10000, 1 << 24)
        values = rng.choice([-1, 0, 0, 1, 1, 1, 2, 3, 6])
        while n * (1 + abs(values)) > 1 << 28:
            n //= 2
        first, end = rng.choice([(0, 32), (0, 32), (0, 32), (0, 24), (0, 16), (7, 25), (24, 32)])
        type = rng.choice(["uint32", "uint32", "float32", "int32"]) if kind == "array" and end - first == 32 else "uint32"
        case = _sort("", n, values, first, end, rng.choice(["uniform", "uniform", "low"]), type, kind)
    del case["name"]
    return case


def _carried(case):
    return 1 if case["values"] == -1 else case["values"]


def _sizes(case):
    """Sizes of the arrays of a batch; the layout belongs to the case."""
    u = np.random.RandomState(case["count"] * 7 + 1).uniform(math.log(case["lo"]),
                                                             math.log(case["hi"] + 1), case["count"])
    return np.clip(np.floor(np.exp(u)).astype(np.int64), case["lo"], case["hi"])


def _total(case):
    return case["n"] if "n" in case else int(_sizes(case).sum())


def _inputs(case, seed):
    """[1 + given value arrays][total] random words: the keys, then the values."""
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)
    n = _total(case)
    words = torch.empty((1 + max(0, case["values"]), n), dtype=torch.int32, device=_DEV)
    words.random_(-(1 << 31), 1 << 31, generator=g)
    if case["type"] == "float32":
        words[0].view(torch.float32).normal_(generator=g)
    elif case["keys"] == "low":  # AND of three words: each bit set once in eight
        for _ in range(2):
            words[0] &= torch.empty_like(words[0]).random_(-(1 << 31), 1 << 31, generator=g)
    if case["end"] == 24 and case["first"] == 0:
        words[0] &= (1 << 24) - 1
    return words


_engine = None


def _get_engine():
    global _engine
    if _engine is None:
        _engine = mg.Engine()
        _engine.set_stream(torch.cuda.current_stream().cuda_stream)
    return _engine


def prepare(case, seed):
    n, carried = _total(case), _carried(case)
    state = {"case": case, "engine": _get_engine(), "source": _inputs(case, seed)}
    rows = 1 + carried
    side0 = torch.empty((rows, n), dtype=torch.int32, device=_DEV)
    state["filled"] = side0[: state["source"].shape[0]]
    state["side0"] = side0
    if case["kind"] == "serve":  # sorted in place: the service has its own scratch
        starts = np.concatenate([[0], np.cumsum(_sizes(case))])
        requests = []
        for i in range(case["count"]):
            r = mg.SortRequest()
            at = int(starts[i]) * 4
            r.keys = side0[0].data_ptr() + at
            for v in range(carried):
                r.values[v] = side0[1 + v].data_ptr() + at
            r.numElements, r.valueCount = int(starts[i + 1] - starts[i]), case["values"]
            r.firstBit, r.endBit = case["first"], case["end"]
            requests.append(r)
        state["requests"], state["arrivals"] = requests, [0.0] * len(requests)
        budget = max(1 << 26, 16 * n * (1 + carried))
        state["server"] = mg.Server(state["engine"], budget, max_in_flight=3, max_elements=1 << 20)
        return state
    side1 = torch.empty((rows, n), dtype=torch.int32, device=_DEV)
    state["side1"] = side1
    d = mg.SortData()
    d.maxElements = d.numElements = n
    d.valueCount, d.firstBit, d.endBit = case["values"], case["first"], case["end"]
    state["data"] = d
    _point(state)
    if case["kind"] == "plan":
        starts = np.concatenate([[0], np.cumsum(_sizes(case))])
        state["plan"] = state["engine"].segmented_plan(d, starts)
    return state


def _point(state):
    """The descriptor with the input on side 0."""
    d, carried = state["data"], _carried(state["case"])
    n = d.numElements
    for side, t in enumerate((state["side0"], state["side1"])):
        at = t.data_ptr()
        d.keys[side] = at
        for v in range(carried):
            d.values[v][side] = at + 4 * n * (1 + v)
    d.parity = 0


def run(state):
    case = state["case"]
    torch.add(state["source"], 0, out=state["filled"])
    if case["kind"] == "serve":
        # The service works on streams of its own: the input has to be there.
        torch.cuda.current_stream().synchronize()
        done = state["server"].replay(state["requests"], state["arrivals"])
        for c in done:
            if c.status != mg.SortStatus.SUCCESS:
                raise mg.MgpuError(c.status, "served request")
        return state["side0"]
    _point(state)
    d, engine = state["data"], state["engine"]
    if case["kind"] == "plan":
        state["plan"].execute(d)
    elif case["kind"] == "ex":
        engine.sort_array_ex(d, 256, 8, 6)
    elif case["type"] != "uint32":
        engine.sort_array_typed(d, _TYPES[case["type"]])
    else:
        engine.sort_array(d)
    return state["side0"] if d.keys[0] == state["side0"].data_ptr() else state["side1"]


def work(case):
    # Keys read and written once; values likewise, generated indices written.
    words = 2 + (1 if case["values"] == -1 else 2 * case["values"])
    return {"bytes": 4.0 * words * _total(case), "flops": 0.0}


def exact(case, seed):
    words = _inputs(case, seed)
    n = words.shape[1]
    key = words[0].to(torch.int64)
    if case["type"] == "float32":
        key = torch.where(key < 0, ~key, key | (1 << 31)) & 0xFFFFFFFF
    elif case["type"] == "int32":
        key = (key ^ (1 << 31)) & 0xFFFFFFFF
    key = (key & 0xFFFFFFFF) >> case["first"] & ((1 << (case["end"] - case["first"])) - 1)
    local = torch.arange(n, device=_DEV)
    if "count" in case:  # each array by itself: the array's number above the field
        sizes = torch.from_numpy(_sizes(case)).to(_DEV)
        key |= torch.repeat_interleave(torch.arange(case["count"], device=_DEV), sizes) << 32
        local -= torch.repeat_interleave(torch.cumsum(sizes, 0) - sizes, sizes)
    order = torch.sort(key, stable=True)[1]
    del key
    rows = [words[0][order]]
    if case["values"] == -1:
        rows.append(local[order].to(torch.int32))
    rows += [words[1 + v][order] for v in range(max(0, case["values"]))]
    return torch.stack(rows)
