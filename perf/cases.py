"""The calls this device system is timed with: what a program built on it has it do, through the
public entry points (thrust_amd.capi, the binding of the C interface), from calls of a few
thousand elements, where launches and host time count, to arrays of a gigabyte and more, which
the memory bounds.

  listed()             twelve calls that stand for the range
  draw(rng)            one more call of the same range, odd sizes among them
  prepare(case, seed)  inputs, output buffers and temporary storage a program has in hand before the call
  run(state)           one pass; returns the call's whole outputs
  work(case)           bytes and operations a pass cannot do without
  tolerance(case)      what another correct implementation at the same precision may differ by

In-place algorithms (the sorts, stable_partition) work on a copy the pass makes of its input, as a
program does that still needs the input: a pass can be repeated, and it always meets unsorted
keys.  Counts of selected elements or runs stay on the device; output buffers start out zeroed, so
that what lies behind the last element of a result is the same everywhere.
"""
import torch

from thrust_amd import capi

_CODES = {"i32": capi.I32, "u32": capi.U32, "f32": capi.F32, "i64": capi.I64, "u64": capi.U64, "f64": capi.F64}
_BYTES = {"i32": 4, "u32": 4, "f32": 4, "i64": 8, "u64": 8, "f64": 8}
_TORCH = {"i32": torch.int32, "u32": torch.int32, "f32": torch.float32,
          "i64": torch.int64, "u64": torch.int64, "f64": torch.float64}


def listed():
    return [
        # the smallest sorts: a frontier, a bucket, one screen's worth of depth keys
        {"name": "sort_i32_3k", "op": "sort", "n": 3_001, "key": "i32"},
        # an ordinary sort: identifiers or hashes of one batch
        {"name": "sort_u32_1m", "op": "sort", "n": 1_000_003, "key": "u32"},
        # the sort this project's headline figure is quoted on
        {"name": "sort_u32_2p28", "op": "sort", "n": 1 << 28, "key": "u32"},
        # an argsort of measurements: float keys around zero that carry their index
        {"name": "sort_pairs_f32_u32_5m", "op": "sort_pairs", "n": 5_000_011, "key": "f32"},
        # the largest sort by key: 64-bit identifiers that carry their index
        {"name": "sort_pairs_u64_u32_2p27", "op": "sort_pairs", "n": 1 << 27, "key": "u64"},
        # a small reduction: a norm, a mean, a check inside an iteration
        {"name": "reduce_f32_100k", "op": "reduce", "n": 100_003, "key": "f32"},
        # the reduction of a whole array
        {"name": "reduce_i32_2p28", "op": "reduce", "n": 1 << 28, "key": "i32"},
        # an ordinary scan: counts to offsets
        {"name": "inclusive_scan_i32_1m", "op": "inclusive_scan", "n": (1 << 20) + 13, "key": "i32"},
        # the scan of a whole array
        {"name": "inclusive_scan_i32_2p28", "op": "inclusive_scan", "n": 1 << 28, "key": "i32"},
        # a group-by sum over sorted keys, runs of eight on average
        {"name": "reduce_by_key_i32_f32_4m", "op": "reduce_by_key", "n": 4_000_037, "key": "i32", "mean_run": 8},
        # a filter over a whole array that keeps half of it
        {"name": "copy_if_f32_half_2p28", "op": "copy_if", "n": 1 << 28, "key": "f32", "keep": 0.5},
        # two sorted batches with payloads joined into one
        {"name": "merge_by_key_u32_u32_2x2m", "op": "merge_by_key", "n": 4_000_038, "key": "u32"},
    ]


# largest drawn size per call and element width: none costs more than the largest listed call
_RANGES = {
    "sort": (("i32", "u32", "f32", "i64", "u64"), 1 << 28, 1 << 27),
    "sort_pairs": (("i32", "u32", "f32", "u64"), 1 << 27, 1 << 26),
    "reduce": (("i32", "u32", "f32", "i64", "f64"), 1 << 28, 1 << 27),
    "inclusive_scan": (("i32", "u32", "f32", "i64"), 1 << 28, 1 << 27),
    "exclusive_scan": (("i32", "u32", "f32", "i64"), 1 << 28, 1 << 27),
    "reduce_by_key": (("i32", "u32"), 1 << 28, 1 << 27),
    "unique_by_key": (("i32", "u32"), 1 << 28, 1 << 27),
    "copy_if": (("i32", "f32", "f64"), 1 << 28, 1 << 27),
    "stable_partition": (("i32", "f32", "f64"), 1 << 28, 1 << 27),
    "merge_by_key": (("i32", "u32", "f32"), 1 << 28, 1 << 27),
}
_SMALLEST = 1_000


def draw(rng):
    op = rng.choice(sorted(_RANGES))
    keys, most_narrow, most_wide = _RANGES[op]
    key = rng.choice(keys)
    most = most_narrow if _BYTES[key] == 4 else most_wide
    n = int(_SMALLEST * (most / _SMALLEST) ** rng.random())
    if rng.random() < 0.75:
        n |= 1  # three in four are odd
    n = min(max(n, _SMALLEST), most)
    case = {"op": op, "n": n, "key": key}
    if op in ("copy_if", "stable_partition"):
        case["keep"] = rng.choice((0.05, 0.5, 0.9))
    elif op in ("reduce_by_key", "unique_by_key"):
        case["mean_run"] = rng.choice((8, 1000))
    return case


def _array(kind, tensor):
    return capi.DeviceArray(tensor.numel(), _CODES[kind], tensor.view(torch.uint8))


def _empty(kind, n):
    return _array(kind, torch.zeros(n, dtype=_TORCH[kind], device="cuda"))


def _full_range(kind, n, gen):
    """Sort keys: integers over their full range, floats around zero with a wide spread."""
    if kind in ("f32", "f64"):
        return torch.randn(n, dtype=_TORCH[kind], device="cuda", generator=gen) * 1000
    if _BYTES[kind] == 4:
        return torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int32, device="cuda", generator=gen)
    high = torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int64, device="cuda", generator=gen)
    return (high << 32) | torch.randint(0, 1 << 32, (n,), dtype=torch.int64, device="cuda", generator=gen)


def _values(kind, n, gen):
    """Numbers to add up or to test: integers in [0, 1000], floats in [0, 1)."""
    if kind in ("f32", "f64"):
        return torch.rand(n, dtype=_TORCH[kind], device="cuda", generator=gen)
    return torch.randint(0, 1001, (n,), dtype=_TORCH[kind], device="cuda", generator=gen)


def _runs(kind, n, mean_run, gen):
    """Sorted keys: the numbers of runs whose lengths are geometric with the given mean."""
    starts = torch.rand(n, device="cuda", generator=gen) < 1.0 / mean_run
    return torch.cumsum(starts, 0, dtype=torch.int32)


def _sorted_keys(kind, n, gen):
    if kind == "u32":  # the order of the unsigned values, not of the signed tensor that holds them
        return torch.sort(_full_range("i32", n, gen))[0] ^ (-(1 << 31))
    return torch.sort(_full_range(kind, n, gen))[0]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    op, n, key = case["op"], case["n"], case["key"]
    state = {"op": op, "key": key, "temp": capi.Temp(), "n": n}
    if op in ("sort", "sort_pairs"):
        state["src"] = _array(key, _full_range(key, n, gen))
        state["work"] = _empty(key, n)
        if op == "sort_pairs":
            state["src_values"] = _array("u32", torch.randperm(n, device="cuda", generator=gen, dtype=torch.int32))
            state["work_values"] = _empty("u32", n)
    elif op == "stable_partition":
        state["src"] = _array(key, _values(key, n, gen))
        state["work"] = _empty(key, n)
    elif op == "reduce":
        state["x"] = _array(key, _values(key, n, gen))
        state["out"] = capi.DeviceArray(1, _CODES[key])
    elif op in ("inclusive_scan", "exclusive_scan", "copy_if"):
        state["x"] = _array(key, _values(key, n, gen))
        state["out"] = _empty(key, n)
    elif op in ("reduce_by_key", "unique_by_key"):
        state["keys"] = _array(key, _runs(key, n, case["mean_run"], gen))
        state["values"] = _array("f32", _values("f32", n, gen))
        state["keys_out"], state["values_out"] = _empty(key, n), _empty("f32", n)
    elif op == "merge_by_key":
        na = n // 2
        state["ka"], state["kb"] = _array(key, _sorted_keys(key, na, gen)), _array(key, _sorted_keys(key, n - na, gen))
        order = torch.randperm(n, device="cuda", generator=gen, dtype=torch.int32)
        state["va"], state["vb"] = _array("u32", order[:na].clone()), _array("u32", order[na:].clone())
        state["keys_out"], state["values_out"] = _empty(key, n), _empty("u32", n)
    if op in ("copy_if", "stable_partition"):
        # integers are uniform in [0, 1000], floats in [0, 1)
        state["threshold"] = case["keep"] if key in ("f32", "f64") else int(round(1001 * case["keep"]))
    return state


def _typed(array, kind):
    return array.storage[:array.n * array.itemsize].view(_TORCH[kind])


def _count(array):
    return array.storage[:8].view(torch.int64)


def _copy(dst, src):
    capi.check(capi.load().thrust_amd_memcpy(dst.ptr, src.ptr, src.n * src.itemsize, capi.D2D, capi.stream_ptr()),
               "thrust_amd_memcpy")


def run(state):
    op, key, temp = state["op"], state["key"], state["temp"]
    if op == "sort":
        _copy(state["work"], state["src"])
        capi.sort_keys(state["work"], temp=temp)
        return _typed(state["work"], key)
    if op == "sort_pairs":
        _copy(state["work"], state["src"])
        _copy(state["work_values"], state["src_values"])
        capi.sort_pairs(state["work"], state["work_values"], temp=temp)
        return _typed(state["work"], key), _typed(state["work_values"], "u32")
    if op == "stable_partition":
        _copy(state["work"], state["src"])
        count = capi.stable_partition(state["work"], capi.LT, state["threshold"], temp=temp, read_count=False)
        return _typed(state["work"], key), _count(count)
    if op == "reduce":
        return _typed(capi.reduce(state["x"], temp=temp, out=state["out"]), key)
    if op == "inclusive_scan":
        return _typed(capi.inclusive_scan(state["x"], out=state["out"], temp=temp), key)
    if op == "exclusive_scan":
        return _typed(capi.exclusive_scan(state["x"], init=0, out=state["out"], temp=temp), key)
    if op == "copy_if":
        out, count = capi.copy_if(state["x"], capi.LT, state["threshold"], out=state["out"], temp=temp, read_count=False)
        return _typed(out, key), _count(count)
    if op == "merge_by_key":
        keys, values = capi.merge_by_key(state["ka"], state["kb"], state["va"], state["vb"], temp=temp,
                                         keys_out=state["keys_out"], values_out=state["values_out"])
        return _typed(keys, key), _typed(values, "u32")
    call = capi.reduce_by_key if op == "reduce_by_key" else capi.unique_by_key
    keys, values, count = call(state["keys"], state["values"], temp=temp, keys_out=state["keys_out"],
                               values_out=state["values_out"], read_count=False)
    return _typed(keys, key), _typed(values, "f32"), _count(count)


def work(case):
    op, n, b = case["op"], case["n"], _BYTES[case["key"]]
    if op == "sort":
        return {"bytes": 2 * b * n, "flops": 0}
    if op in ("sort_pairs", "merge_by_key"):
        return {"bytes": 2 * (b + 4) * n, "flops": 0}
    if op == "stable_partition":
        return {"bytes": 2 * b * n, "flops": n}
    if op == "reduce":
        return {"bytes": b * n, "flops": n}
    if op in ("inclusive_scan", "exclusive_scan"):
        return {"bytes": 2 * b * n, "flops": n}
    if op == "copy_if":
        return {"bytes": int(b * n * (1 + case["keep"])), "flops": n}
    return {"bytes": int((b + 4) * n * (1 + 1 / case["mean_run"])), "flops": n}  # reduce_by_key, unique_by_key


def tolerance(case):
    # Bit-exact except sums of floats, whose order of addition is free: about four times what the path
    # differs by from the same sums in 64 bits (from the same sum backwards for f64), over 1e4 to 2^28 elements:
    # reduce 7.4e-8 and 1.8e-16, scans 5.4e-7, run sums 9.9e-8.
    if case["op"] == "reduce" and case["key"] in ("f32", "f64"):
        return {"rel": 3e-7 if case["key"] == "f32" else 1e-15}
    if case["op"] in ("inclusive_scan", "exclusive_scan") and case["key"] == "f32":
        return {"rel": 2e-6}
    if case["op"] == "reduce_by_key":
        return {"rel": 4e-7}
    return "exact"
