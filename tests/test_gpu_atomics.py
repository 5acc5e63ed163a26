"""GPU parity: bulk atomics (histogram by fetch_add, strided fetch ops).

Final contents must be bit-exact against the oracle's serial fold
(order-independent operations) for both the privatized and the global
strategy.
"""
import ctypes

import numpy as np
import pytest

import opensycl_amd as acpp
import oracle as O
from gpu_util import dev, host, rand, zipf_keys

pytestmark = pytest.mark.gpu

STRATS = [acpp.ATOMICS_PRIVATIZED, acpp.ATOMICS_GLOBAL, acpp.ATOMICS_AUTO]


# 4096 bins keep 8 LDS copies of each counter, 8192 bins 4, 16384 bins 2,
# 32768 one; above that the counters are packed 16-bit
@pytest.mark.parametrize("num_bins", [1, 100, 4096, 8192, 16384, 32768, 32769, 65536])
@pytest.mark.parametrize("strategy", STRATS)
def test_histogram_zipf(gpu, q, scratch, num_bins, strategy):
    torch, _ = gpu
    for n in (1, 1001, (1 << 22) + 3):
        keys = zipf_keys(n, num_bins + 10, seed=n)  # some keys out of range
        start = rand(np.uint32, num_bins, seed=1, lo=0, hi=1000)
        bins = dev(torch, start)
        acpp.histogram(q, scratch, dev(torch, keys), bins, strategy)
        q.wait()
        assert np.array_equal(host(bins), O.histogram(keys, num_bins, start)), (n, strategy)


@pytest.mark.parametrize("num_bins", [4096, 65536])
def test_histogram_hot_bins_drain(gpu, q, scratch, num_bins):
    # every key in bin 0 or bin 1: the 16-bit LDS fields cross 0x8000 many
    # times per work-group and must drain without carrying into a neighbour
    torch, _ = gpu
    n = 1 << 24
    for hot in (0, 1, num_bins - 1):
        keys = np.full(n, hot, dtype=np.uint32)
        keys[::7] = (hot + 1) % num_bins
        bins = torch.zeros(num_bins, dtype=torch.uint32, device="cuda")
        acpp.histogram(q, scratch, dev(torch, keys), bins, acpp.ATOMICS_PRIVATIZED)
        q.wait()
        assert np.array_equal(host(bins), O.histogram(keys, num_bins)), hot


def test_histogram_misaligned_keys(gpu, q, scratch):
    torch, _ = gpu
    keys = zipf_keys(1000003, 4096, seed=3)
    for off in (1, 2, 3):
        kd = dev(torch, keys)[off:]
        for strat in (acpp.ATOMICS_PRIVATIZED, acpp.ATOMICS_GLOBAL):
            bins = torch.zeros(4096, dtype=torch.uint32, device="cuda")
            acpp.histogram(q, scratch, kd, bins, strat)
            q.wait()
            assert np.array_equal(host(bins), O.histogram(keys[off:], 4096))


# Above 65536 bins the bins are cut into 2 .. 64 slices (2^22 bins); one bin
# more takes one atomic per key.  2^17 keys are the last that need no scratch.
@pytest.mark.parametrize("num_bins", [65537, 131072, 131073, 200000, 1 << 20, (1 << 20) + 1, 1 << 22, (1 << 22) + 1])
@pytest.mark.parametrize("n", [1, 4097, 1 << 17, (1 << 17) + 1, (1 << 22) + 3])
def test_histogram_sliced(gpu, q, scratch, num_bins, n):
    torch, _ = gpu
    rng = np.random.default_rng(n)
    skewed = zipf_keys(n, num_bins + 10, seed=n)  # some keys out of range
    spread = rng.integers(0, num_bins + 100, n).astype(np.uint32)
    strided = (np.arange(n, dtype=np.uint64) * 4096 % num_bins).astype(np.uint32)
    one = np.full(n, num_bins - 1, dtype=np.uint32)  # its 16-bit counter drains
    for keys in (skewed, spread, strided, one):
        for off in (0, 1):
            start = rand(np.uint32, num_bins, seed=1, lo=0, hi=1000)
            bins = dev(torch, start)
            acpp.histogram(q, scratch, dev(torch, keys)[off:], bins)
            q.wait()
            scratch.release()
            assert np.array_equal(host(bins), O.histogram(keys[off:], num_bins, start)), off


@pytest.mark.parametrize("num_bins", [4096, 65536, 200000])
def test_histogram_captured(gpu, num_bins):
    # replays add to the bins like eager calls; the sliced form captures
    # without scratch
    torch, _ = gpu
    n = (1 << 20) + 7
    keys = zipf_keys(n, num_bins, seed=9)
    kd = dev(torch, keys)
    bins = torch.zeros(num_bins, dtype=torch.uint32, device="cuda")
    cache = acpp.AllocationCache()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        q = acpp.Queue()
        with acpp.AllocationGroup(cache) as scratch:
            if num_bins <= 65536:  # leaves the scratch in the cache
                acpp.histogram(q, scratch, kd, bins)
                q.wait()
        scratch = acpp.AllocationGroup(cache)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            acpp.histogram(acpp.Queue(), scratch, kd, bins)
        calls = 1 if num_bins <= 65536 else 0
        once = O.histogram(keys, num_bins).astype(np.uint64)
        for _ in range(3):
            graph.replay()
            with acpp.AllocationGroup(cache) as other:
                acpp.histogram(q, other, kd, bins)
                q.wait()
            calls += 2
            assert np.array_equal(host(bins), (once * calls).astype(np.uint32))
    del graph
    scratch.close()
    cache.close()


@pytest.mark.parametrize("dtype", [np.int32, np.uint32, np.int64, np.uint64, np.float32,
                                   np.float64])
@pytest.mark.parametrize("num_slots", [1, 64, 1000, 1024, 4096, 70000])
def test_strided_fetch_ops(gpu, q, scratch, dtype, num_slots):
    torch, _ = gpu
    n = (1 << 20) + 5
    if np.issubdtype(dtype, np.floating):
        # small integers: every partial sum stays below 2^24, so float sums
        # are exact in any order
        v = np.round(rand(np.float64, n, seed=num_slots) * 4).astype(dtype)
    else:
        v = rand(dtype, n, seed=num_slots, lo=-(1 << 20) if np.iinfo(dtype).min < 0 else 0,
                 hi=1 << 20)
    idx = (np.arange(n) % num_slots).astype(np.uint32)
    for op in ("max", "min", "add"):
        for strat in STRATS:
            if strat == acpp.ATOMICS_PRIVATIZED and num_slots * v.itemsize > 128 * 1024:
                continue
            start = np.zeros(num_slots, dtype=dtype) + dtype(3)
            t = dev(torch, start)
            acpp.atomic_fetch_strided(q, scratch, op, dev(torch, v), t, strat)
            q.wait()
            exp = start.copy()
            if op == "max":
                np.maximum.at(exp, idx, v)
            elif op == "min":
                np.minimum.at(exp, idx, v)
            else:
                np.add.at(exp, idx, v)
            assert np.array_equal(host(t), exp), (op, strat)


def test_fetch_max_i32_oracle(gpu, q, scratch):
    # The atomics workload shape: uniform int32 into 1024 slots, slot = i mod 1024
    torch, _ = gpu
    n = 1 << 24
    v = rand(np.int32, n, seed=11)
    for strat in STRATS:
        t = torch.full((1024,), np.iinfo(np.int32).min, dtype=torch.int32, device="cuda")
        acpp.atomic_fetch_strided(q, scratch, "max", dev(torch, v), t, strat)
        q.wait()
        assert np.array_equal(host(t), O.fetch_max_strided(v, 1024)), strat
    # misaligned view -> head elements through the scalar path
    t = torch.full((1024,), np.iinfo(np.int32).min, dtype=torch.int32, device="cuda")
    acpp.atomic_fetch_strided(q, scratch, "max", dev(torch, v)[3:], t, acpp.ATOMICS_PRIVATIZED)
    q.wait()
    assert np.array_equal(host(t), O.fetch_max_strided(v[3:], 1024))


@pytest.mark.parametrize("dtype", [np.int32, np.int64, np.float32])
def test_strided_lds_form_misaligned_view(gpu, q, scratch, dtype):
    # 1000 slots do not divide the work-group stride: the LDS form, with a
    # view 3 elements into the buffer (scalar head, then 16-byte loads)
    torch, _ = gpu
    n = (1 << 21) + 9
    v = np.round(rand(np.float64, n + 3, seed=5) * 4).astype(dtype)
    vd = dev(torch, v)[3:]
    idx = (np.arange(n) % 1000).astype(np.uint32)
    for op in ("max", "min", "add"):
        start = np.zeros(1000, dtype=dtype) + dtype(3)
        t = dev(torch, start)
        acpp.atomic_fetch_strided(q, scratch, op, vd, t, acpp.ATOMICS_PRIVATIZED)
        q.wait()
        exp = start.copy()
        {"max": np.maximum, "min": np.minimum, "add": np.add}[op].at(exp, idx, v[3:])
        assert np.array_equal(host(t), exp), op


# Strips of 64 columns of 16 bytes (256 above 160 MiB), rows repeated to at
# least 512 columns: slot counts around those edges, fewer elements than
# slots, fewer rows than a group's bands, views, and a group size that is no
# power of two.
@pytest.mark.parametrize("dtype", [np.int32, np.float32, np.float64])
@pytest.mark.parametrize("num_slots", [1, 3, 255, 256, 257, 2047, 2049, 32769, 65537])
def test_strided_strips(gpu, q, scratch, dtype, num_slots):
    torch, _ = gpu
    for n in (1, 5, num_slots - 1, num_slots, num_slots + 1, 3 * num_slots + 2, (1 << 18) + 7):
        if n < 1:
            continue
        # small integers: float sums are exact in any order
        v = np.round(rand(np.float64, n + 3, seed=num_slots) * 4).astype(dtype)
        vd = dev(torch, v)
        for off in (0, 1, 3):
            x = v[off:off + n]
            idx = np.arange(n) % num_slots
            for op, fold in (("add", np.add), ("min", np.minimum), ("max", np.maximum)):
                for cfg in (None, (192,)):
                    t = torch.full((num_slots,), 3, dtype=vd.dtype, device="cuda")
                    acpp.atomic_fetch_strided(q, scratch, op, vd[off:off + n], t, config=cfg)
                    q.wait()
                    exp = np.zeros(num_slots, dtype=dtype) + dtype(3)
                    fold.at(exp, idx, x)
                    assert np.array_equal(host(t), exp), (n, off, op, cfg)


def test_strided_strips_wide(gpu, q, scratch):
    # above 160 MiB a strip is 256 columns wide and streams past the caches
    torch, _ = gpu
    n = (1 << 26) + 1003
    for num_slots in (1000, 40000):
        v = (torch.arange(n, device="cuda") % 7 - 3).to(torch.float32)
        t = torch.zeros(num_slots, dtype=torch.float32, device="cuda")
        acpp.atomic_fetch_strided(q, scratch, "add", v, t)
        q.wait()
        rows = n // num_slots
        exp = v[:rows * num_slots].view(rows, num_slots).double().sum(0)
        exp[:n - rows * num_slots] += v[rows * num_slots:]
        assert torch.equal(t.double(), exp), num_slots


# Rows of a little more than two strips are replaced by longer ones (18, 33, 50
# and 130 slots of fp32) where the values are enough for four bands of them;
# few slots are folded in steps of four.
@pytest.mark.parametrize("num_slots", [1, 3, 17, 18, 33, 50, 130, 513])
@pytest.mark.parametrize("n", [1 << 15, (1 << 21) + 5, 160 * (1 << 18) - 1, 160 * (1 << 18) + 3])
def test_strided_long_rows(gpu, q, scratch, num_slots, n):
    torch, _ = gpu
    rows = n // num_slots
    v = (torch.arange(n, device="cuda") % 7 - 3).to(torch.float32)  # sums are exact in any order
    for op in ("add", "max"):
        t = torch.full((num_slots,), -5.0, dtype=torch.float32, device="cuda")
        acpp.atomic_fetch_strided(q, scratch, op, v, t)
        q.wait()
        whole, rest = v[:rows * num_slots].view(rows, num_slots), v[rows * num_slots:]
        if op == "add":
            exp = whole.double().sum(0) - 5
            exp[:rest.numel()] += rest
        else:
            exp = whole.max(0).values.double()
            exp[:rest.numel()] = torch.maximum(exp[:rest.numel()], rest.double())
        assert torch.equal(t.double(), exp), op


# Plain counters added straight to the bins (up to 8192 bins; up to 32768 for
# at most 5 x 2^17 keys and 3 x 2^20 counters in all groups), and the packed
# ones with partials beyond.
@pytest.mark.parametrize("num_bins", [1, 63, 64, 65, 127, 500, 1747, 8192, 8193, 16001, 19660, 19661, 32768, 32769])
def test_histogram_direct_flush_whole_waves(gpu, q, scratch, num_bins):
    torch, _ = gpu
    for n in (1, 4097, 1 << 17, (1 << 17) + 1, 5 << 17, (5 << 17) + 1, 1 << 20):
        keys = (torch.arange(n, device="cuda") * 7919 % (num_bins + 2)).to(torch.int32)  # two out of range
        bins = torch.full((num_bins,), 9, dtype=torch.int32, device="cuda")
        acpp.histogram(q, scratch, keys.view(torch.uint32), bins.view(torch.uint32))
        q.wait()
        exp = torch.bincount(keys.long(), minlength=num_bins)[:num_bins] + 9
        assert torch.equal(bins.long(), exp), n


def _order_dependent(got, start, v, idx, num_slots, op):
    """Float fetch_min / fetch_max: slots without a NaN hold the exact result;
    in a slot with one, whatever the order of its elements, the result is that
    NaN or one of the slot's numbers (numbers before the NaN, the start value
    among them, do not survive it)."""
    exp = np.where(np.isnan(start) & (np.arange(num_slots) < len(v)), -np.inf if op == "max" else np.inf, start)
    with np.errstate(invalid="ignore"):
        (np.maximum if op == "max" else np.minimum).at(exp, idx, v)  # propagates NaN
    clean = ~np.isnan(exp)
    assert np.array_equal(got[clean], exp[clean]), op
    for s in np.flatnonzero(~clean):
        assert np.isnan(got[s]) or got[s] in v[idx == s], (op, s, got[s])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n, num_slots", [(5, 3), (70, 64), (1500, 1000), (5000, 4093), (100003, 70000),
                                          ((1 << 16) + 3, 7), ((1 << 20) + 1, 600)])
def test_strided_fetch_min_max_nan_and_infinities(gpu, q, scratch, dtype, n, num_slots):
    # A NaN as the last element of a slot, in slots of one and of many
    # elements; infinities of both signs; slots of the operator's worst values.
    torch, _ = gpu
    v = np.round(rand(np.float64, n, seed=n) * 4).astype(dtype)
    idx = (np.arange(n) % num_slots).astype(np.uint32)
    last = n - 1 - (n - 1 - np.arange(min(num_slots, n))) % num_slots
    v[last[::3]] = np.nan
    v[np.arange(1, n, 7)] = np.inf
    v[np.arange(2, n, 11)] = -np.inf
    for op, worst in (("max", -np.inf), ("min", np.inf)):
        for offset in (0, 1):
            w = v.copy()
            w[idx == 1] = worst  # nothing but the identity
            start = np.full(num_slots, 1e30 if op == "max" else -1e30, dtype=dtype)
            start[1] = worst
            start[2::5] = np.nan  # gives way to the slot's elements
            t = dev(torch, start)
            buf = dev(torch, np.concatenate([np.zeros(offset, dtype=dtype), w]))[offset:]
            acpp.atomic_fetch_strided(q, scratch, op, buf, t)
            q.wait()
            _order_dependent(host(t), start, w, idx, num_slots, op)


def test_strided_fetch_add_keeps_negative_zero(gpu, q, scratch):
    torch, _ = gpu
    for n, num_slots in ((10, 3), (5000, 64), (100003, 70000)):
        t = torch.full((num_slots,), -0.0, device="cuda")
        acpp.atomic_fetch_strided(q, scratch, "add", torch.full((n,), -0.0, device="cuda"), t)
        q.wait()
        assert bool(torch.signbit(t).all()), (n, num_slots)


def _graph_nodes(graph):
    hip = ctypes.CDLL("libamdhip64.so")
    nodes = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(nodes)) == 0
    return nodes.value


@pytest.mark.parametrize("warm", [True, False])
@pytest.mark.parametrize("num_bins, n", [(40000, 1 << 24), (65536, 1 << 24), (65537, 1 << 22), (200000, 1 << 22)])
def test_captured_histogram_takes_cached_partials(gpu, q, num_bins, n, warm):
    # Where the cache holds the scratch of an earlier call, a captured call of
    # bins that fit one LDS goes through partials as that one did (a counting
    # and a combining kernel); else, and with more bins, it needs no scratch (the
    # counting kernel alone).
    torch, _ = gpu
    keys = rand(np.uint32, n, seed=num_bins) % np.uint32(num_bins)
    kd = dev(torch, keys)
    cache = acpp.AllocationCache()
    scratch = acpp.AllocationGroup(cache)
    bins = torch.zeros(num_bins, dtype=torch.int32, device="cuda").view(torch.uint32)
    if warm:
        acpp.histogram(q, scratch, kd, bins)
        q.wait()
        scratch.release()
    s = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=s):
        acpp.histogram(acpp.Queue(), scratch, kd, bins)
    assert _graph_nodes(graph) == (2 if warm and num_bins <= 65536 else 1)
    graph.instantiate()
    once = O.histogram(keys, num_bins).astype(np.uint64)
    for calls in (1, 2, 3):
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(bins), (once * (calls + warm)).astype(np.uint32))
    del graph
    scratch.close()
    cache.close()


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint), ("y", ctypes.c_uint), ("z", ctypes.c_uint)]


class _KernelNode(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", _Dim3),
                ("args", ctypes.c_void_p), ("lds", ctypes.c_uint)]


def _first_kernel(graph):
    hip = ctypes.CDLL("libamdhip64.so")
    g, count = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t(8)
    nodes = (ctypes.c_void_p * 8)()
    assert hip.hipGraphGetNodes(g, nodes, ctypes.byref(count)) == 0 and count.value >= 1
    params = _KernelNode()
    assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(nodes[0]), ctypes.byref(params)) == 0
    return params


@pytest.mark.parametrize("num_bins, n, wg, lds, block, most_groups", [
    (65537, 2048, 0, False, None, None),    # few keys, more bins than one LDS: one atomic per key
    (1 << 22, 4096, 0, False, None, None),
    (200000, 4097, 0, True, 1024, None),    # slices from here on
    (65537, 2049, 0, True, 1024, None),
    (300000, 100000, 64, True, 1024, None),  # slices are 1024 wide whatever is asked for
    (300000, 1000, 64, False, 64, None),
    (60000, 100000, 256, True, 256, None),
    (150, 1_000_000, 0, True, 1024, 96),    # few bins: no more groups than flush in the time of the keys
    (150, 300_000, 0, True, 1024, 74),
    (8192, 3_000_000, 0, True, 1024, 245),
])
def test_histogram_forms(gpu, num_bins, n, wg, lds, block, most_groups):
    torch, _ = gpu
    keys = rand(np.uint32, n, seed=n) % np.uint32(num_bins + 3)
    kd = dev(torch, keys)
    bins = torch.zeros(num_bins, dtype=torch.int32, device="cuda").view(torch.uint32)
    cache = acpp.AllocationCache()
    scratch = acpp.AllocationGroup(cache)
    s = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=s):
        acpp.histogram(acpp.Queue(), scratch, kd, bins, config={"work_group_size": wg} if wg else None)
    kernel = _first_kernel(graph)
    assert (kernel.lds > 0) == lds
    if block:
        assert kernel.block.x == block
    if most_groups:
        assert kernel.grid.x in (most_groups * block, most_groups)  # in work-items or work-groups
    graph.instantiate()
    graph.replay()
    torch.cuda.synchronize()
    assert np.array_equal(host(bins), O.histogram(keys, num_bins))
    del graph
    scratch.close()
    cache.close()


@pytest.mark.parametrize("num_bins", [8193, 9000, 12000, 20001, 32767, 32768, 32769, 40001, 65535, 65536, 65537, 200001])
@pytest.mark.parametrize("wg", [0, 64, 192])
def test_histogram_flushes_in_many_rounds(gpu, q, scratch, num_bins, wg):
    # few keys straight to the bins, several words a round; every bin is hit
    # and those next to the end are not
    torch, _ = gpu
    rng = np.random.default_rng(num_bins)
    for n in (1, 5000, num_bins + 1, 130000):
        keys = np.concatenate([np.arange(num_bins - 1, -1, -1), rng.integers(0, num_bins + 2, n)])[:n].astype(np.uint32)
        bins = torch.full((num_bins + 64,), 9, dtype=torch.int32, device="cuda").view(torch.uint32)
        acpp.histogram(q, scratch, dev(torch, keys), bins[:num_bins],
                       config={"work_group_size": wg} if wg else None)
        q.wait()
        got = host(bins)
        assert np.array_equal(got[:num_bins], O.histogram(keys, num_bins) + np.uint32(9)), n
        assert np.all(got[num_bins:] == 9), n


@pytest.mark.parametrize("dtype, num_slots, wg, n, groups", [
    (np.float64, 35982, 0, 2_000_000, 564),   # 282 strips on 256 CUs: two groups each
    (np.float64, 35982, 0, 100_000, 71),      # a row and a bit, in wider strips
    (np.int64, 200, 64, 8_000_000, 510),      # two narrow groups a CU
    (np.int64, 200, 64, 24_000_000, 1530),    # six: the cache does not hold the input
    (np.int32, 4096, 192, 42_000_000, 768),
    (np.int32, 200, 64, 8_000_000, 504),
    (np.int64, 200, 512, 8_000_000, 250),
])
def test_strided_groups(gpu, dtype, num_slots, wg, n, groups):
    torch, _ = gpu
    v = rand(dtype, n, seed=n, lo=-1000, hi=1000) if np.issubdtype(dtype, np.integer) else \
        np.round(rand(np.float64, n, seed=n) * 100)
    vd = dev(torch, v)
    t = dev(torch, np.full(num_slots, 3, dtype=dtype))
    cache = acpp.AllocationCache()
    scratch = acpp.AllocationGroup(cache)
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        acpp.atomic_fetch_strided(acpp.Queue(), scratch, "max", vd, t, config={"work_group_size": wg} if wg else None)
    assert _first_kernel(graph).grid.x == groups
    graph.instantiate()
    graph.replay()
    torch.cuda.synchronize()
    exp = np.full(num_slots, 3, dtype=dtype)
    np.maximum.at(exp, np.arange(n) % num_slots, v)
    assert np.array_equal(host(t), exp)
    del graph
    scratch.close()
    cache.close()
