"""Python mirror of ``acpp::algorithms`` (include/hipSYCL/algorithms/numeric.hpp).

Every function has the reference's argument order -- queue, scratch
allocation group, input range, output, init, operator -- with torch device
tensors standing for the iterator ranges.  Calls are asynchronous on the
queue's stream, like the reference's (doc/algorithms.md:35-37); use
``queue.wait()`` before reading results on the host.

The device work is done by the HIP library through its C-ABI
(``opensycl_amd._abi``); nothing here computes on the CPU.
"""
from __future__ import annotations

import ctypes
import struct
from typing import Optional

from . import _abi
from ._abi import LaunchConfig, check

# Operator codes (== __acpp_sscp_algorithm_op, builtin_config.hpp:27-37)
PLUS = 0
MULTIPLY = 1
MIN = 2
MAX = 3
BIT_AND = 4
BIT_OR = 5
BIT_XOR = 6
LOGICAL_AND = 7
LOGICAL_OR = 8

_OP_NAMES = {
    "plus": PLUS, "multiplies": MULTIPLY, "multiply": MULTIPLY, "minimum": MIN, "min": MIN,
    "maximum": MAX, "max": MAX, "bit_and": BIT_AND, "bit_or": BIT_OR, "bit_xor": BIT_XOR,
    "logical_and": LOGICAL_AND, "logical_or": LOGICAL_OR,
}

# Element transform codes (acpp_unary_op): the unary callables of
# transform_reduce and the transform scans (numeric.hpp:193-212, 299-327).
IDENTITY = 0
NEGATE = 1
ABS = 2
SQUARE = 3
TWICE = 4
BIT_NOT = 5
IS_ZERO = 6
IS_NONZERO = 7

_UNARY_NAMES = {
    "identity": IDENTITY, "negate": NEGATE, "abs": ABS, "square": SQUARE, "twice": TWICE,
    "bit_not": BIT_NOT, "is_zero": IS_ZERO, "is_nonzero": IS_NONZERO,
}

ALLOCATION_DEVICE = 0
ALLOCATION_SHARED = 1
ALLOCATION_HOST = 2


def _torch():
    import torch
    return torch


# What the calls look up, filled on first use: a short call spends more time
# here than on the device (1000 int32 elements scanned in a group of their own:
# 6.9 us a call, 5.6 us with these tables and the pooled groups below).
_tags: dict = {}        # dtype -> tag
_functions: dict = {}   # (name, dtype) -> library function


def _tag(dtype) -> str:
    if not _tags:
        torch = _torch()
        _tags.update({
            torch.int8: "i8", torch.int16: "i16", torch.int32: "i32", torch.int64: "i64",
            torch.uint8: "u8", torch.uint16: "u16", torch.uint32: "u32", torch.uint64: "u64",
            torch.float32: "f32", torch.float64: "f64", torch.bfloat16: "bf16",
        })
    tag = _tags.get(dtype)
    if tag is None:
        raise TypeError(f"unsupported element type {dtype}")
    return tag


def _function(name: str, dtype):
    """The library's function `name`_<tag of dtype>."""
    fn = _functions.get((name, dtype))
    if fn is None:
        fn = getattr(_abi.load(), f"{name}_{_tag(dtype)}")
        _functions[(name, dtype)] = fn
    return fn


def _op(op) -> int:
    if isinstance(op, str):
        if op not in _OP_NAMES:
            raise ValueError(f"unknown operator {op!r}")
        return _OP_NAMES[op]
    return int(op)


def _unary(transform) -> int:
    if isinstance(transform, str):
        if transform not in _UNARY_NAMES:
            raise ValueError(f"unknown element transform {transform!r}")
        return _UNARY_NAMES[transform]
    return int(transform)


def _cfg(config):
    if config is None:
        return None
    if isinstance(config, LaunchConfig):
        return ctypes.byref(config)
    if isinstance(config, dict):
        return ctypes.byref(LaunchConfig(**config))
    wg, ipt, gpc, flags = (tuple(config) + (0, 0, 0, 0))[:4]
    return ctypes.byref(LaunchConfig(wg, ipt, gpc, flags))


class Queue:
    """In-order queue on a HIP stream (torch stream or raw hipStream_t)."""

    def __init__(self, stream=None, device: int = 0):
        torch = _torch()
        self.device = device
        if stream is None:
            stream = torch.cuda.current_stream(device)
        self.stream = stream

    @property
    def handle(self) -> int:
        s = self.stream
        return s if isinstance(s, int) else s.cuda_stream

    def wait(self) -> None:
        """Wait for the queue's work, then raise the device's asynchronous
        errors (queue::wait_and_throw, include/hipSYCL/sycl/queue.hpp:
        378-383): AcppError with status ERROR_WATCHDOG if a kernel gave up
        waiting for another work-group, whose results are then wrong."""
        if isinstance(self.stream, int):
            _torch().cuda.synchronize(self.device)
        else:
            self.stream.synchronize()
        check_asynchronous_errors(self.device)


def check_asynchronous_errors(device: int = 0) -> None:
    """acpp_check_asynchronous_errors: raise (once) for a watchdog give-up
    on `device` since the last check.  Non-blocking: synchronise first."""
    check(_abi.load().acpp_check_asynchronous_errors(device))


class AllocationCache:
    """util::allocation_cache (allocation_cache.hpp:42-127)."""

    def __init__(self, allocation_type: int = ALLOCATION_DEVICE):
        lib = _abi.load()
        h = ctypes.c_void_p()
        check(lib.acpp_allocation_cache_create(allocation_type, ctypes.byref(h)))
        self._h = h
        self._owned = [h]        # until it is destroyed
        self._groups: dict = {}  # device -> handles of closed (empty) groups, for new ones
        self._alive: dict = {}   # the library's groups on this cache, open or in _groups
        self._closing = False

    @property
    def handle(self):
        return None if self._closing else self._h

    def purge(self) -> None:
        self._destroy_groups()
        check(_abi.load().acpp_allocation_cache_purge(self._h))

    def _destroy_groups(self) -> None:
        for pool in list(self._groups.values()):
            try:
                while True:
                    self._destroy_group(pool.pop())
            except IndexError:  # empty, maybe because another thread took the last one
                pass

    def _destroy_group(self, h) -> int:
        st = _abi.load().acpp_allocation_group_destroy(h)
        self._alive.pop(h.value, None)
        if self._closing:
            self._destroy()
        return st

    def _destroy(self) -> None:
        if self._alive:
            return
        try:
            h = self._owned.pop()  # (one step: two threads may close the last two groups)
        except IndexError:
            return
        self._h = None
        check(_abi.load().acpp_allocation_cache_destroy(h))

    def close(self) -> None:
        """Free the cache.  Groups that are still open return their regions to
        it: it is freed with the last of them (the garbage collector may
        finalise a cache before its groups)."""
        if self._h and not self._closing:
            self._destroy_groups()
            self._closing = True
            self._destroy()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class AllocationGroup:
    """util::allocation_group (allocation_cache.hpp:142-181)."""

    def __init__(self, cache: AllocationCache, device: int = 0):
        pool = cache._groups.get(device)
        try:
            h = pool.pop()  # (one step: other threads may take from the pool)
        except (AttributeError, IndexError):
            h = ctypes.c_void_p()
            check(_abi.load().acpp_allocation_group_create(cache.handle, device, ctypes.byref(h)))
            cache._alive[h.value] = None
            pool = cache._groups.setdefault(device, [])
        self._h = h
        self._cache = cache
        self._pool = pool           # where close() leaves the handle
        self._plans = 0             # live SegmentedPlans made from this group
        self._close_pending = False

    @property
    def handle(self):
        return self._h

    def obtain(self, nbytes: int, alignment: int = 256) -> int:
        p = ctypes.c_void_p()
        check(_abi.load().acpp_allocation_group_obtain(self._h, nbytes, alignment,
                                                       ctypes.byref(p)))
        return p.value

    def release(self) -> None:
        """Return the group's regions to the cache now.  Refused while a
        SegmentedPlan made from this group is alive: it still
        uses them, and replays would corrupt whichever call got them next."""
        if self._plans > 0:
            raise RuntimeError("AllocationGroup.release: a SegmentedPlan made from this group is alive; "
                               "close the plan first")
        check(_abi.load().acpp_allocation_group_release(self._h))

    def watchdog_trips(self) -> int:
        """Look-backs that gave up waiting in the scratch regions this group
        holds (blocking; call after the group's work has completed).  A
        non-zero count means some results are wrong; expected to be 0."""
        v = ctypes.c_uint64()
        check(_abi.load().acpp_allocation_group_watchdog_trips(self._h, ctypes.byref(v)))
        return v.value

    def close(self) -> None:
        """Return the group's regions to the cache.  While a SegmentedPlan
        made from this group is alive, it still uses them: the
        release then waits until the last such plan is closed."""
        if self._plans > 0:
            self._close_pending = True
            return
        if self._h:
            h, self._h = self._h, None
            # emptied even when it reports an asynchronous error
            if not self._cache._closing and len(self._pool) < 16:
                st = _abi.load().acpp_allocation_group_release(h)
                self._pool.append(h)
            else:
                st = self._cache._destroy_group(h)
            if st:
                check(st)

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def compute_units(device: int = 0) -> int:
    v = ctypes.c_int()
    check(_abi.load().acpp_device_compute_units(device, ctypes.byref(v)))
    return v.value


def _ptr(t) -> int:
    if t is None:
        return 0
    if not t.is_cuda:
        raise ValueError("tensors must live in device memory")
    return t.data_ptr()


def _check_contig(*ts):
    for t in ts:
        if t is not None and not t.is_contiguous():
            raise ValueError("tensors must be contiguous")


def _check_out(out, dtype, count: int, what: str) -> None:
    """The C-ABI receives raw pointers only, so an output too short or of a
    narrower type would be written past its end: reject it before launch."""
    if out is None:
        raise ValueError(f"{what}: output is missing")
    if out.dtype != dtype:
        raise TypeError(f"{what}: output must be {dtype}, not {out.dtype}")
    if out.numel() < count:
        raise ValueError(f"{what}: output holds {out.numel()} elements, needs {count}")


def _acc_dtype(x):
    """Result type of a reduction over x: float32 for bf16 input."""
    torch = _torch()
    return torch.float32 if x.dtype == torch.bfloat16 else x.dtype


def _scalar(tag: str, v):
    if type(v) is int and -2**31 <= v < 2**31:
        return v  # the argument's own type converts it
    ct = _abi.SCALAR_TAGS.get(tag, ctypes.c_float)
    return ct(v)


def reduce(q: Queue, scratch: AllocationGroup, x, out, init=0, op=PLUS, config=None) -> None:
    """algorithms::reduce (numeric.hpp:226-249): out[0] = op(init, fold(x))."""
    _check_contig(x, out)
    _check_out(out, _acc_dtype(x), 1, "reduce")
    tag = _tag(x.dtype)
    fn = _function("acpp_reduce", x.dtype)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(out), _scalar(tag, init),
             _op(op), _cfg(config)))


def reduce_compensated(q: Queue, scratch: AllocationGroup, x, out, init=0.0,
                       config=None) -> None:
    """Compensated fp32 sum of fp32 or bf16 input into an fp32 out[0]."""
    _check_contig(x, out)
    tag = _tag(x.dtype)
    if tag not in ("f32", "bf16"):
        raise TypeError("compensated sums take float32 or bfloat16 input")
    _check_out(out, _torch().float32, 1, "reduce_compensated")
    fn = _function("acpp_reduce_compensated", x.dtype)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(out), ctypes.c_float(init),
             _cfg(config)))


# Pair transform codes of the binary transform_reduce (== acpp_binary_op)
B_MULTIPLIES, B_PLUS, B_MINUS, B_ABS_DIFF, B_SQ_DIFF, B_MIN, B_MAX, B_BIT_AND, B_BIT_OR, B_BIT_XOR = range(10)
_BINARY_NAMES = {
    "multiplies": B_MULTIPLIES, "plus": B_PLUS, "minus": B_MINUS, "abs_diff": B_ABS_DIFF,
    "sq_diff": B_SQ_DIFF, "minimum": B_MIN, "maximum": B_MAX, "bit_and": B_BIT_AND, "bit_or": B_BIT_OR,
    "bit_xor": B_BIT_XOR,
}


def transform_reduce(q: Queue, scratch: AllocationGroup, x1, x2, out, init=0,
                     compensated: bool = False, config=None, reduce_op=PLUS,
                     transform=B_MULTIPLIES) -> None:
    """Binary transform_reduce (numeric.hpp:170-223): out[0] = reduce_op(init,
    reduce_op over transform(x1[i], x2[i])).  The default (plus, multiplies)
    is the dot product, also for bf16 and in the compensated form; other
    pairs (reduce_op: plus, multiplies, minimum, maximum; transform: a pair
    transform code or name) take 32/64-bit integers, float32 and float64."""
    _check_contig(x1, x2, out)
    if x1.numel() > x2.numel() or x1.dtype != x2.dtype:
        raise ValueError("second range must have the first range's type and length")
    tag = _tag(x1.dtype)
    _check_out(out, _torch().float32 if compensated else _acc_dtype(x1), 1, "transform_reduce")
    code = _BINARY_NAMES[transform] if isinstance(transform, str) else int(transform)
    op = _op(reduce_op)
    lib = _abi.load()
    if (op, code) != (PLUS, B_MULTIPLIES):
        if compensated or tag == "bf16":
            raise TypeError("compensated and bf16 transform_reduce take plus with multiplies only")
        fn = _function("acpp_transform_reduce_binary", x1.dtype)
        check(fn(scratch.handle, q.handle, _ptr(x1), x1.numel(), _ptr(x2), _ptr(out), _scalar(tag, init), op,
                 code, _cfg(config)))
        return
    if compensated:
        if tag not in ("f32", "bf16"):
            raise TypeError("compensated dot products take float32 or bfloat16 input")
        fn = _function("acpp_transform_reduce_dot_compensated", x1.dtype)
        init_c = ctypes.c_float(init)
    else:
        fn = _function("acpp_transform_reduce_dot", x1.dtype)
        init_c = ctypes.c_float(init) if tag == "bf16" else _scalar(tag, init)
    check(fn(scratch.handle, q.handle, _ptr(x1), x1.numel(), _ptr(x2), _ptr(out), init_c,
             _cfg(config)))


def transform_reduce_unary(q: Queue, scratch: AllocationGroup, x, out, init=0, op=PLUS,
                           transform=IDENTITY, config=None) -> None:
    """Unary transform_reduce (numeric.hpp:193-212):
    out[0] = op(init, fold_op(transform(x[i]))); empty x leaves out as is."""
    _check_contig(x, out)
    _check_out(out, x.dtype, 1, "transform_reduce")
    tag = _tag(x.dtype)
    fn = _function("acpp_transform_reduce", x.dtype)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(out), _scalar(tag, init),
             _op(op), _unary(transform), _cfg(config)))


def reduction(q: Queue, scratch: AllocationGroup, x, out, op=PLUS,
              initialize_to_identity: bool = False, config=None, identity=None) -> None:
    """parallel_for(range{n}, sycl::reduction(out, [identity,] op
    [, initialize_to_identity])) whose kernel combines x[i]
    (reduction.hpp:165-236): with initialize_to_identity out[0] = op(identity,
    fold), else op(out[0], fold).  Without a given identity the operator's
    own is used."""
    _check_contig(x, out)
    _check_out(out, x.dtype, 1, "reduction")
    flag = 1 if initialize_to_identity else 0
    if identity is None:
        fn = _function("acpp_reduction", x.dtype)
        check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(out), _op(op), flag, _cfg(config)))
    else:
        fn = _function("acpp_reduction_identity", x.dtype)
        check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(out), _scalar(_tag(x.dtype), identity),
                 _op(op), flag, _cfg(config)))


# Host arrays of up to four pointers or ints, as bytes.
_pointers = [struct.Struct(f"@{k}P") for k in range(5)]
_ints = [struct.Struct(f"@{k}i") for k in range(5)]


def reduction_multi(q: Queue, scratch: AllocationGroup, inputs, outs, ops,
                    initialize_to_identity=False, config=None, identities=None) -> None:
    """Up to four sycl::reduction objects in one parallel_for
    (handler.hpp:799-975): outs[k][0] = fold of inputs[k] with ops[k]
    (starting from the identity, or from outs[k][0]).  Inputs share one
    length and element type; they may be the same tensor.
    initialize_to_identity: one flag for all, or one per reduction;
    identities: None, or one given identity per reduction."""
    k = len(inputs)
    if not (1 <= k <= 4) or len(outs) != k or len(ops) != k:
        raise ValueError("one to four (input, output, operator) triples")
    n = inputs[0].numel()
    tag = _tag(inputs[0].dtype)
    dtype = inputs[0].dtype
    for x, o in zip(inputs, outs):
        _check_contig(x, o)
        if x.numel() != n or x.dtype != dtype or o.dtype != dtype:
            raise ValueError("inputs must share length and element type with the outputs")
        _check_out(o, x.dtype, 1, "reduction_multi")
    arr_in = _pointers[k].pack(*[_ptr(x) for x in inputs])
    arr_out = _pointers[k].pack(*[_ptr(o) for o in outs])
    arr_ops = _ints[k].pack(*[_op(o) for o in ops])
    if identities is None and isinstance(initialize_to_identity, bool):
        fn = _function("acpp_reduction_multi", inputs[0].dtype)
        check(fn(scratch.handle, q.handle, k, arr_in, n, arr_out, arr_ops, int(initialize_to_identity),
                 _cfg(config)))
        return
    flags = list(initialize_to_identity) if not isinstance(initialize_to_identity, bool) \
        else [initialize_to_identity] * k
    if len(flags) != k or (identities is not None and len(identities) != k):
        raise ValueError("one initialize_to_identity flag and identity per reduction")
    arr_flags = _ints[k].pack(*[int(bool(f)) for f in flags])
    arr_id = None
    if identities is not None:
        ct = _abi.SCALAR_TAGS[tag]
        arr_id = (ct * k)(*identities)
    fn = _function("acpp_reduction_multi_identity", inputs[0].dtype)
    check(fn(scratch.handle, q.handle, k, arr_in, n, arr_out, arr_ops, arr_id, arr_flags, _cfg(config)))


def inclusive_scan(q: Queue, scratch: AllocationGroup, x, d, op=PLUS, init=None,
                   config=None) -> None:
    """algorithms::inclusive_scan (numeric.hpp:253-279)."""
    _check_contig(x, d)
    _check_out(d, x.dtype, x.numel(), "inclusive_scan")
    tag = _tag(x.dtype)
    fn = _function("acpp_inclusive_scan", x.dtype)
    init_p = None
    if init is not None:
        init_c = _abi.SCALAR_TAGS[tag](init)
        init_p = ctypes.addressof(init_c)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(d), _op(op), init_p,
             _cfg(config)))


def exclusive_scan(q: Queue, scratch: AllocationGroup, x, d, init=0, op=PLUS,
                   config=None) -> None:
    """algorithms::exclusive_scan (numeric.hpp:281-297)."""
    _check_contig(x, d)
    _check_out(d, x.dtype, x.numel(), "exclusive_scan")
    tag = _tag(x.dtype)
    fn = _function("acpp_exclusive_scan", x.dtype)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(d), _scalar(tag, init),
             _op(op), _cfg(config)))


def transform_inclusive_scan(q: Queue, scratch: AllocationGroup, x, d, op=PLUS,
                             transform=IDENTITY, init=None, config=None) -> None:
    """algorithms::transform_inclusive_scan (numeric.hpp:299-317): the
    inclusive scan of transform(x[i])."""
    _check_contig(x, d)
    _check_out(d, x.dtype, x.numel(), "transform_inclusive_scan")
    tag = _tag(x.dtype)
    fn = _function("acpp_transform_inclusive_scan", x.dtype)
    init_p = None
    if init is not None:
        init_c = _abi.SCALAR_TAGS[tag](init)
        init_p = ctypes.addressof(init_c)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(d), _op(op), _unary(transform),
             init_p, _cfg(config)))


def transform_exclusive_scan(q: Queue, scratch: AllocationGroup, x, d, init=0, op=PLUS,
                             transform=IDENTITY, config=None) -> None:
    """algorithms::transform_exclusive_scan (numeric.hpp:319-327): the
    exclusive scan of transform(x[i]) starting from init."""
    _check_contig(x, d)
    _check_out(d, x.dtype, x.numel(), "transform_exclusive_scan")
    tag = _tag(x.dtype)
    fn = _function("acpp_transform_exclusive_scan", x.dtype)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(d), _scalar(tag, init),
             _op(op), _unary(transform), _cfg(config)))


# ---------------------------------------------------------------------------
# Bulk atomics (atomic_ref fetch_add / fetch_min / fetch_max in a loop)
# ---------------------------------------------------------------------------
ATOMICS_AUTO = 0
ATOMICS_PRIVATIZED = 1
ATOMICS_GLOBAL = 2


def histogram(q: Queue, scratch: AllocationGroup, keys, bins, strategy: int = ATOMICS_AUTO,
              config=None) -> None:
    """bins[k] += number of keys equal to k (keys >= len(bins) are ignored)."""
    _check_contig(keys, bins)
    if _tag(keys.dtype) != "u32" or _tag(bins.dtype) != "u32":
        raise TypeError("histogram takes uint32 keys and uint32 bins")
    check(_abi.load().acpp_histogram_u32(scratch.handle, q.handle, _ptr(keys), keys.numel(),
                                         _ptr(bins), bins.numel(), strategy, _cfg(config)))


def atomic_fetch_strided(q: Queue, scratch: AllocationGroup, op: str, values, target,
                         strategy: int = ATOMICS_AUTO, config=None) -> None:
    """target[i % len(target)] = op(target[i % len(target)], values[i]) for op in
    add / min / max."""
    _check_contig(values, target)
    if op not in ("add", "min", "max"):
        raise ValueError("op must be add, min or max")
    if values.dtype != target.dtype:
        raise TypeError("values and target must have the same type")
    if target.numel() < 1:
        raise ValueError("target must hold at least one slot")
    fn = _function(f"acpp_atomic_fetch_{op}_strided", values.dtype)
    check(fn(scratch.handle, q.handle, _ptr(values), values.numel(), _ptr(target), target.numel(),
             strategy, _cfg(config)))


# ---------------------------------------------------------------------------
# copy_if (stream compaction)
# ---------------------------------------------------------------------------
PRED_NONZERO, PRED_EQ, PRED_NE, PRED_LT, PRED_LE, PRED_GT, PRED_GE, PRED_MASK_EQ = range(8)


_COPY_IF_TAGS = ("i8", "u8", "i16", "u16", "i32", "u32", "i64", "u64", "f32", "f64")


def copy_if(q: Queue, scratch: AllocationGroup, x, d, pred: int, operand=0, mask=0, num_copied=None,
            config=None) -> None:
    """algorithms::copy_if (algorithm.hpp:178-243) with a data predicate:
    d[0..count) = the x[i] with pred(x[i]); num_copied[0] = count (a uint64
    device tensor, optional)."""
    _check_contig(x, d)
    _check_out(d, x.dtype, x.numel(), "copy_if")
    if num_copied is not None:
        _check_out(num_copied, _torch().uint64, 1, "copy_if num_copied")
    tag = _tag(x.dtype)
    if tag not in _COPY_IF_TAGS:
        raise TypeError(f"copy_if takes integer, f32 or f64 elements, not {tag}")
    fn = _function("acpp_copy_if", x.dtype)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(d), int(pred), _scalar(tag, operand),
             _scalar(tag, mask), _ptr(num_copied) if num_copied is not None else None, _cfg(config)))


def copy_if_stencil(q: Queue, scratch: AllocationGroup, x, stencil, d, num_copied=None,
                    config=None) -> None:
    """copy_if with the predicate evaluated by the caller: copies x[i] where
    stencil[i] != 0 (stencil: uint8 or bool tensor of x's length)."""
    _check_contig(x, d, stencil)
    if stencil.numel() < x.numel() or stencil.element_size() != 1:
        raise ValueError("stencil must be a one-byte tensor at least as long as x")
    _check_out(d, x.dtype, x.numel(), "copy_if_stencil")
    if num_copied is not None:
        _check_out(num_copied, _torch().uint64, 1, "copy_if_stencil num_copied")
    tag = _tag(x.dtype)
    if tag not in _COPY_IF_TAGS:
        raise TypeError(f"copy_if takes integer, f32 or f64 elements, not {tag}")
    fn = _function("acpp_copy_if_stencil", x.dtype)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(stencil), _ptr(d),
             _ptr(num_copied) if num_copied is not None else None, _cfg(config)))


# ---------------------------------------------------------------------------
# Segmented scans and reductions
# ---------------------------------------------------------------------------
def _seg_check(x, offsets):
    if _tag(offsets.dtype) != "u64":
        raise TypeError("offsets must be uint64")
    if offsets.numel() < 1:
        raise ValueError("offsets must hold num_segments + 1 entries")
    _check_contig(x, offsets)


def segmented_inclusive_scan(q: Queue, scratch: AllocationGroup, x, d, offsets, op=PLUS,
                             config=None) -> None:
    """d[i] = inclusive scan of x within the segment [offsets[s], offsets[s+1])."""
    _seg_check(x, offsets)
    _check_contig(d)
    _check_out(d, x.dtype, x.numel(), "segmented_inclusive_scan")
    tag = _tag(x.dtype)
    fn = _function("acpp_segmented_inclusive_scan", x.dtype)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(d), _ptr(offsets),
             offsets.numel() - 1, _op(op), _cfg(config)))


def segmented_reduce(q: Queue, scratch: AllocationGroup, x, offsets, out, init=0, op=PLUS,
                     config=None) -> None:
    """out[s] = op(init, fold of x over [offsets[s], offsets[s+1]))."""
    _seg_check(x, offsets)
    _check_contig(out)
    _check_out(out, x.dtype, offsets.numel() - 1, "segmented_reduce")
    tag = _tag(x.dtype)
    fn = _function("acpp_segmented_reduce", x.dtype)
    check(fn(scratch.handle, q.handle, _ptr(x), x.numel(), _ptr(offsets), offsets.numel() - 1,
             _ptr(out), _scalar(tag, init), _op(op), _cfg(config)))


class SegmentedPlan:
    """A segmented scan or reduction whose scratch and parameters are kept
    for every ``launch``.

    The plan holds raw pointers to the input, output and offsets
    tensors and to scratch regions of the allocation group, so the plan
    keeps references to all of them (and to the group's cache) for as long
    as it lives: a launch never touches freed or reissued memory.  Launches
    of one plan share that scratch: they have to be ordered on the device
    (one stream, or events between streams); launches that may overlap need
    plans of their own."""

    def __init__(self, handle, scratch, keep=()):
        self._h = handle
        self._scratch = scratch
        scratch._plans += 1
        self._keep = tuple(keep)

    @staticmethod
    def inclusive_scan(scratch: AllocationGroup, x, d, offsets, op=PLUS, config=None):
        _seg_check(x, offsets)
        _check_contig(d)
        _check_out(d, x.dtype, x.numel(), "segmented plan inclusive_scan")
        tag = _tag(x.dtype)
        h = ctypes.c_void_p()
        fn = _function("acpp_segmented_plan_inclusive_scan", x.dtype)
        check(fn(scratch.handle, _ptr(x), x.numel(), _ptr(d), _ptr(offsets), offsets.numel() - 1,
                 _op(op), _cfg(config), ctypes.byref(h)))
        return SegmentedPlan(h, scratch, (x, d, offsets))

    @staticmethod
    def reduce(scratch: AllocationGroup, x, offsets, out, init=0, op=PLUS, config=None):
        _seg_check(x, offsets)
        _check_contig(out)
        _check_out(out, x.dtype, offsets.numel() - 1, "segmented plan reduce")
        tag = _tag(x.dtype)
        h = ctypes.c_void_p()
        fn = _function("acpp_segmented_plan_reduce", x.dtype)
        check(fn(scratch.handle, _ptr(x), x.numel(), _ptr(offsets), offsets.numel() - 1,
                 _ptr(out), _scalar(tag, init), _op(op), _cfg(config), ctypes.byref(h)))
        return SegmentedPlan(h, scratch, (x, out, offsets))

    def launch(self, q: Queue) -> None:
        check(_abi.load().acpp_segmented_plan_launch(self._h, q.handle))

    def close(self) -> None:
        if self._h:
            h, self._h = self._h, None
            check(_abi.load().acpp_segmented_plan_destroy(h))
        self._keep = ()
        g, self._scratch = self._scratch, None
        if g is not None:
            g._plans -= 1
            if g._close_pending and g._plans == 0:
                g.close()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass
