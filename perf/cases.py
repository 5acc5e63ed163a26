"""The calls that programs make of this library, as cases that can be timed.

Each case is one call (or, where the library adds to its target, the clear
that a program puts before it) through the Python interface, on inputs that
are resident in device memory: device-wide scans, reductions and dot
products, stream compaction, segmented scans and sums, histograms and strided
atomic updates.  ``listed()`` holds the fixed ones, ``draw()`` more of the
same ranges.
"""
import functools

import torch

import opensycl_amd as acpp

_TYPES = {
    "i8": torch.int8, "i16": torch.int16, "i32": torch.int32, "i64": torch.int64,
    "f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16,
}
_SIZES = {"i8": 1, "i16": 2, "bf16": 2, "i32": 4, "f32": 4, "i64": 8, "f64": 8}


def listed():
    return [
        # A short prefix sum inside a larger program (offsets of a small
        # batch): what one call costs when there is almost nothing to do.
        {"name": "scan_i32_1k", "path": "scan", "type": "i32", "n": 1000, "exclusive": True, "op": "plus", "offset": 0},
        # An ordinary ragged scan whose data fits the caches.
        {"name": "scan_f32_1m", "path": "scan", "type": "f32", "n": 1048583, "exclusive": False, "op": "plus",
         "offset": 0},
        # The bandwidth-bound scan of the benchmark's headline step.
        {"name": "scan_i32_256m", "path": "scan", "type": "i32", "n": 1 << 28, "exclusive": True, "op": "plus",
         "offset": 0},
        # A running peak over 16-bit samples, from a buffer that starts one
        # sample after an allocation's start (a view x[1:]).
        {"name": "peak_i16_20m", "path": "transform_scan", "type": "i16", "n": 20000003, "exclusive": False,
         "op": "max", "transform": "abs", "offset": 1},
        # The sum of an ordinary, ragged array.
        {"name": "sum_f32_3m", "path": "reduce", "type": "f32", "n": 3000017, "op": "plus", "compensated": False,
         "offset": 0},
        # The dot product of the benchmark's headline step.
        {"name": "dot_f32_256m", "path": "dot", "type": "f32", "n": 1 << 28, "compensated": False, "offset": 0},
        # Filtering a medium-sized column by a threshold.
        {"name": "filter_i32_5m", "path": "copy_if", "type": "i32", "n": 5000011, "keep": 0.5, "stencil": False,
         "offset": 0},
        # The segmented workload of the benchmark: 65,536 segments of very
        # uneven (log-normal) lengths, through a plan that is kept.
        {"name": "segscan_i64_64k", "path": "segmented_scan", "type": "i64", "n": 245953805, "segments": 65536,
         "sigma": 2.0, "plan": True, "offset": 0},
        # Sums of the rows of a batch: few, long, ragged segments.
        {"name": "rowsum_f32_48", "path": "segmented_reduce", "type": "f32", "n": 50000021, "segments": 48,
         "sigma": 0.5, "plan": False, "offset": 0},
        # The larger histogram of the benchmark: Zipf(1.1) keys, 65,536 bins.
        {"name": "hist_zipf_64k", "path": "histogram", "n": 1 << 26, "bins": 65536, "zipf": 1.1, "offset": 0},
        # Counting how often each of 200,000 ids (of a vocabulary, a user
        # table) occurs in a batch of them.
        {"name": "hist_zipf_200k", "path": "histogram", "n": 33554467, "bins": 200000, "zipf": 1.1, "offset": 0},
        # Column sums of a 4,000 x 30,000 matrix by strided fetch_add.
        {"name": "colsum_f32_30k", "path": "fetch", "type": "f32", "n": 120000000, "slots": 30000, "op": "add",
         "offset": 0},
    ]


def draw(rng):
    def size(low, high):  # log-uniform, so mostly odd values
        return max(1, int(2.0 ** rng.uniform(low, high)))

    def top(kind):  # at most 2^28 elements and 1 GiB
        return min(28.0, 30.0 - {1: 0, 2: 1, 4: 2, 8: 3}[_SIZES[kind]])

    path = rng.choice(["scan", "transform_scan", "reduce", "dot", "multi", "copy_if", "segmented_scan",
                       "segmented_reduce", "histogram", "fetch"])
    # one call in four works on a view that starts inside an allocation
    case = {"path": path, "offset": rng.choice([0, 0, 0, rng.randint(1, 3)])}
    if path in ("scan", "transform_scan"):
        case["type"] = rng.choice(["i8", "i16", "i32", "i32", "i64", "f32", "f32", "f64"])
        case["n"] = size(10, top(case["type"]))
        case["exclusive"] = rng.random() < 0.5
        case["op"] = rng.choice(["plus", "plus", "max"])
        if path == "transform_scan":
            case["transform"] = rng.choice(["abs", "negate"])
    elif path == "reduce":
        case["type"] = rng.choice(["i8", "i16", "i32", "i64", "f32", "f32", "f64", "bf16"])
        case["n"] = size(10, top(case["type"]))
        case["op"] = "plus" if case["type"] == "bf16" else rng.choice(["plus", "plus", "max"])
        case["compensated"] = case["type"] in ("f32", "bf16") and case["op"] == "plus" and rng.random() < 0.5
    elif path == "dot":
        case["type"] = rng.choice(["f32", "f32", "f64", "bf16", "i32"])
        case["n"] = size(10, top(case["type"]))
        case["compensated"] = case["type"] in ("f32", "bf16") and rng.random() < 0.5
    elif path == "multi":
        case["type"] = rng.choice(["i32", "f32", "f64"])
        case["n"] = size(10, top(case["type"]) - 1)
    elif path == "copy_if":
        case["type"] = rng.choice(["i8", "i16", "i32", "i32", "i64", "f32", "f64"])
        case["n"] = size(10, top(case["type"]))
        case["keep"] = round(rng.uniform(0.02, 0.98), 3)
        case["stencil"] = rng.random() < 0.4
    elif path in ("segmented_scan", "segmented_reduce"):
        case["type"] = rng.choice(["i32", "i64", "f32", "f64"])
        case["n"] = size(12, top(case["type"]) - 0.1)
        case["segments"] = min(case["n"] // 4, size(0, 24))
        case["sigma"] = rng.choice([0.5, 2.0])
        case["plan"] = rng.random() < 0.5
    elif path == "histogram":
        case["bins"] = size(4, 20)
        case["n"] = size(12, 26 if case["bins"] <= 65536 else 25)
        case["zipf"] = rng.choice([0.0, 1.1])
    else:
        case["type"] = rng.choice(["i32", "i64", "f32", "f64"])
        case["n"] = size(12, top(case["type"]) - 1)
        case["slots"] = min(case["n"] // 2, size(4, 18))
        case["op"] = rng.choice(["add", "add", "max"])
    return case


@functools.lru_cache(maxsize=None)
def _cache():
    """The scratch pool that a program keeps for all its calls."""
    return acpp.AllocationCache()


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _view(t, offset):
    """t's values in a view that starts `offset` elements into an allocation."""
    if not offset:
        return t
    whole = torch.empty(t.numel() + offset, dtype=t.dtype, device=t.device)
    whole[offset:].copy_(t)
    return whole[offset:]


def _values(kind, n, gen, offset=0):
    dtype = _TYPES[kind]
    if dtype.is_floating_point:
        # mean 0.5, deviation 1: both signs, and sums that do not cancel
        x = torch.randn(n, dtype=torch.float64 if kind == "f64" else torch.float32, device="cuda", generator=gen)
        return _view(x.add_(0.5).to(dtype), offset)
    lim = 100 if kind == "i8" else 1000
    return _view(torch.randint(-lim, lim + 1, (n,), dtype=dtype, device="cuda", generator=gen), offset)


def _offsets(case, gen):
    """segments + 1 offsets: log-normal lengths that add up to n (some may be empty)."""
    s, n = case["segments"], case["n"]
    z = torch.randn(s, dtype=torch.float64, device="cuda", generator=gen)
    ends = torch.cumsum(torch.exp(case["sigma"] * z), 0)
    ends = torch.floor(ends * (n / ends[-1])).to(torch.int64).clamp_(0, n)
    ends[-1] = n
    return torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), ends])


def _keys(case, gen):
    """uint32 keys below `bins`, uniform or with P(k) falling as (k + 1)^-zipf."""
    n, bins, s = case["n"], case["bins"], case["zipf"]
    u = torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)
    if s:
        e = 1.0 - s
        u.mul_((bins + 1.0) ** e - 1.0).add_(1.0).pow_(1.0 / e).sub_(1.0)
    else:
        u.mul_(float(bins))
    return u.to(torch.int32).clamp_(0, bins - 1)


def _inputs(case, seed):
    """The input tensors of a case, in signed types."""
    gen = _generator(seed)
    path, off = case["path"], case["offset"]
    if path == "histogram":
        return {"keys": _view(_keys(case, gen), off)}
    if path.startswith("segmented"):
        offsets = _offsets(case, gen)
        return {"x": _values(case["type"], case["n"], gen, off), "offsets": offsets}
    got = {"x": _values(case["type"], case["n"], gen, off)}
    if path == "dot":
        got["y"] = _values(case["type"], case["n"], gen)
    if path == "copy_if" and case["stencil"]:
        got["stencil"] = (torch.rand(case["n"], device="cuda", generator=gen) < case["keep"]).to(torch.uint8)
    return got


def _threshold(case):
    """The value below which about `keep` of a column's values lie."""
    if _TYPES[case["type"]].is_floating_point:
        return 0.5 + float(2 ** 0.5 * torch.erfinv(torch.tensor(2.0 * case["keep"] - 1.0, dtype=torch.float64)))
    lim = 100 if case["type"] == "i8" else 1000
    return int(round((2 * lim + 1) * case["keep"])) - lim


def prepare(case, seed):
    got = _inputs(case, seed)
    path, n = case["path"], case["n"]
    q = acpp.Queue()
    x = got.get("x")
    state = {"inputs": got}
    if path in ("scan", "transform_scan"):
        d = _view(torch.empty(n, dtype=x.dtype, device="cuda"), case["offset"])
        state["out"] = d
        if path == "scan" and case["exclusive"]:
            state["call"] = lambda g: acpp.exclusive_scan(q, g, x, d, 0, case["op"])
        elif path == "scan":
            state["call"] = lambda g: acpp.inclusive_scan(q, g, x, d, case["op"])
        elif case["exclusive"]:
            state["call"] = lambda g: acpp.transform_exclusive_scan(q, g, x, d, 0, case["op"], case["transform"])
        else:
            state["call"] = lambda g: acpp.transform_inclusive_scan(q, g, x, d, case["op"], case["transform"])
    elif path == "reduce":
        out = torch.zeros(1, dtype=torch.float32 if case["type"] == "bf16" else x.dtype, device="cuda")
        state["out"] = out
        if case["compensated"]:
            state["call"] = lambda g: acpp.reduce_compensated(q, g, x, out)
        else:
            state["call"] = lambda g: acpp.reduce(q, g, x, out, 0, case["op"])
    elif path == "dot":
        y = got["y"]
        out = torch.zeros(1, dtype=torch.float32 if case["type"] == "bf16" else x.dtype, device="cuda")
        state["out"] = out
        state["call"] = lambda g: acpp.transform_reduce(q, g, x, y, out, 0, compensated=case["compensated"])
    elif path == "multi":
        # sum, minimum and maximum of one array in one launch
        outs = [torch.zeros(1, dtype=x.dtype, device="cuda") for _ in range(3)]
        state["out"] = outs
        state["call"] = lambda g: acpp.reduction_multi(q, g, [x, x, x], outs, ["plus", "min", "max"], True)
    elif path == "copy_if":
        d = torch.zeros(n, dtype=x.dtype, device="cuda")
        count = torch.zeros(1, dtype=torch.uint64, device="cuda")
        state["out"] = [d, count]
        if case["stencil"]:
            state["call"] = lambda g: acpp.copy_if_stencil(q, g, x, got["stencil"], d, count)
        else:
            bound = _threshold(case)
            state["call"] = lambda g: acpp.copy_if(q, g, x, d, acpp.PRED_LT, bound, num_copied=count)
    elif path in ("segmented_scan", "segmented_reduce"):
        offsets = got["offsets"].view(torch.uint64)
        scan = path == "segmented_scan"
        out = torch.zeros(n if scan else case["segments"], dtype=x.dtype, device="cuda")
        state["out"] = out
        if case["plan"]:
            scratch = acpp.AllocationGroup(_cache())
            if scan:
                plan = acpp.SegmentedPlan.inclusive_scan(scratch, x, out, offsets)
            else:
                plan = acpp.SegmentedPlan.reduce(scratch, x, offsets, out)
            state["plan"], state["queue"], state["scratch"] = plan, q, scratch
        elif scan:
            state["call"] = lambda g: acpp.segmented_inclusive_scan(q, g, x, out, offsets)
        else:
            state["call"] = lambda g: acpp.segmented_reduce(q, g, x, offsets, out)
    elif path == "histogram":
        keys = got["keys"].view(torch.uint32)
        counts = torch.zeros(case["bins"], dtype=torch.int32, device="cuda")
        bins = counts.view(torch.uint32)
        state["out"], state["clear"] = counts, counts
        state["call"] = lambda g: acpp.histogram(q, g, keys, bins)
    else:
        target = torch.zeros(case["slots"], dtype=x.dtype, device="cuda")
        state["out"], state["clear"] = target, target
        state["call"] = lambda g: acpp.atomic_fetch_strided(q, g, case["op"], x, target)
    return state


def run(state):
    if "plan" in state:
        state["plan"].launch(state["queue"])
        return state["out"]
    if "clear" in state:  # the library adds to what the target holds
        state["clear"].zero_()
    with acpp.AllocationGroup(_cache()) as scratch:
        state["call"](scratch)
    return state["out"]


def _kept(case, got):
    return got["stencil"] != 0 if case["stencil"] else got["x"] < _threshold(case)


def work(case):
    path, n = case["path"], case["n"]
    es = _SIZES[case.get("type", "i32")]
    if path in ("scan", "transform_scan"):
        return {"bytes": 2 * n * es, "flops": n}
    if path == "reduce":
        return {"bytes": n * es, "flops": n}
    if path == "dot":
        return {"bytes": 2 * n * es, "flops": 2 * n}
    if path == "multi":
        return {"bytes": n * es, "flops": 3 * n}
    if path == "copy_if":
        return {"bytes": n * es + int(n * case["keep"]) * es + (n if case["stencil"] else 0), "flops": n}
    if path == "segmented_scan":
        return {"bytes": 2 * n * es + 8 * (case["segments"] + 1), "flops": n}
    if path == "segmented_reduce":
        return {"bytes": n * es + (8 + es) * (case["segments"] + 1), "flops": n}
    if path == "histogram":
        return {"bytes": 4 * n + 4 * case["bins"], "flops": n}
    return {"bytes": n * es + es * case["slots"], "flops": n}


def _wide(t):
    return t.double() if t.is_floating_point() else t.to(torch.int64)


def _as(t, like):
    """64-bit values as the type of a whole-number output (wrapping), or in 64 bits."""
    return t if t.is_floating_point() else t.to(like)


def exact(case, seed):
    got = _inputs(case, seed)
    path, n = case["path"], case["n"]
    if path == "histogram":
        return torch.bincount(got["keys"], minlength=case["bins"]).to(torch.int32)
    x = got["x"]
    dtype = x.dtype
    if path == "copy_if":
        keep = _kept(case, got)
        d = torch.zeros(n, dtype=dtype, device="cuda")
        chosen = x[keep]
        d[:chosen.numel()] = chosen
        return [_as(_wide(d), dtype), torch.tensor([chosen.numel()], dtype=torch.int64)]
    w = _wide(x)
    if path in ("scan", "transform_scan"):
        if path == "transform_scan":
            # the transform's result is an element again: it wraps as the type does
            w = _wide((x.abs() if case["transform"] == "abs" else -x))
        w = torch.cumsum(w, 0) if case["op"] == "plus" else torch.cummax(w, 0).values
        if case["exclusive"]:
            first = torch.zeros(1, dtype=w.dtype, device="cuda")
            w = torch.cat([first, w[:-1] if case["op"] == "plus" else w[:-1].clamp_(min=0)])
        return _as(w, dtype)
    if path == "reduce":
        if case["op"] == "max":
            return _as(w.max().clamp(min=0).reshape(1), dtype)
        return _as(w.sum().reshape(1), dtype)
    if path == "dot":
        return _as((w * _wide(got["y"])).sum().reshape(1), dtype)
    if path == "multi":
        return [_as(v.reshape(1), dtype) for v in (w.sum(), w.min(), w.max())]
    if path in ("segmented_scan", "segmented_reduce"):
        offsets = got["offsets"]
        sums = torch.cat([torch.zeros(1, dtype=w.dtype, device="cuda"), torch.cumsum(w, 0)])
        before = sums[offsets[:-1]]
        if path == "segmented_reduce":
            return _as(sums[offsets[1:]] - before, dtype)
        return _as(sums[1:] - torch.repeat_interleave(before, offsets[1:] - offsets[:-1]), dtype)
    # a whole number of rows, then the rest of one
    slots = case["slots"]
    rows = n // slots
    body, rest = w[:rows * slots].view(rows, slots), w[rows * slots:]
    if case["op"] == "max":
        out = body.max(0).values.clamp_(min=0)
        out[:rest.numel()] = torch.maximum(out[:rest.numel()], rest)
    else:
        out = body.sum(0)
        out[:rest.numel()] += rest
    return _as(out, dtype)
