"""Argument checks of the Python mirror (CPU only: nothing is launched).

The C-ABI receives raw pointers and element counts, so an output that is
too short or of a narrower type would be written past its end on the GPU.
The Python functions must reject such outputs before any library call; the
tensors here live on the CPU, so reaching the library would fail
differently (a ValueError about device memory is raised only after these
checks)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import opensycl_amd as acpp  # noqa: E402
from opensycl_amd import algorithms  # noqa: E402


def t(n, dtype=torch.int32):
    return torch.zeros(n, dtype=dtype)


CASES = [
    # (call, expected exception)
    (lambda: acpp.inclusive_scan(None, None, t(10), t(9)), ValueError),
    (lambda: acpp.inclusive_scan(None, None, t(10), t(10, torch.int64)), TypeError),
    (lambda: acpp.exclusive_scan(None, None, t(10, torch.int64), t(10, torch.int32)), TypeError),
    (lambda: acpp.exclusive_scan(None, None, t(10), t(3)), ValueError),
    (lambda: acpp.transform_inclusive_scan(None, None, t(10), t(9)), ValueError),
    (lambda: acpp.transform_exclusive_scan(None, None, t(10), t(10, torch.int16)), TypeError),
    (lambda: acpp.reduce(None, None, t(10), t(0)), ValueError),
    (lambda: acpp.reduce(None, None, t(10, torch.int64), t(1, torch.int32)), TypeError),
    (lambda: acpp.reduce(None, None, t(10, torch.bfloat16), t(1, torch.bfloat16)), TypeError),
    (lambda: acpp.reduce_compensated(None, None, t(10, torch.float32), t(1, torch.float64)), TypeError),
    (lambda: acpp.transform_reduce(None, None, t(10, torch.bfloat16), t(10, torch.bfloat16),
                                   t(1, torch.bfloat16)), TypeError),
    (lambda: acpp.transform_reduce(None, None, t(10, torch.float32), t(10, torch.float32),
                                   t(0, torch.float32), compensated=True), ValueError),
    (lambda: acpp.transform_reduce(None, None, t(10), t(9), t(1)), ValueError),
    (lambda: acpp.transform_reduce_unary(None, None, t(10), t(1, torch.int8)), TypeError),
    (lambda: acpp.reduction(None, None, t(10), t(0)), ValueError),
    (lambda: acpp.reduction_multi(None, None, [t(10)], [t(0)], [acpp.PLUS]), ValueError),
    (lambda: acpp.copy_if(None, None, t(10), t(9), acpp.PRED_NONZERO), ValueError),
    (lambda: acpp.copy_if(None, None, t(10), t(10), acpp.PRED_NONZERO,
                          num_copied=t(1, torch.int64)), TypeError),
    (lambda: acpp.copy_if_stencil(None, None, t(10), t(10, torch.uint8), t(10, torch.int64)), TypeError),
    (lambda: acpp.segmented_inclusive_scan(None, None, t(10), t(9), t(3, torch.uint64)), ValueError),
    (lambda: acpp.segmented_reduce(None, None, t(10), t(5, torch.uint64), t(3)), ValueError),
    (lambda: acpp.segmented_reduce(None, None, t(10), t(0, torch.uint64), t(3)), ValueError),
    (lambda: acpp.atomic_fetch_strided(None, None, "max", t(10), t(0)), ValueError),
    (lambda: acpp.SegmentedPlan.inclusive_scan(None, t(10), t(10, torch.int64), t(3, torch.uint64)),
     TypeError),
    (lambda: acpp.SegmentedPlan.reduce(None, t(10), t(5, torch.uint64), t(2)), ValueError),
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_bad_outputs_are_rejected_before_launch(i):
    call, exc = CASES[i]
    with pytest.raises(exc) as info:
        call()
    assert "device memory" not in str(info.value)


def test_well_formed_call_reaches_the_device_check():
    # the same call with a good output gets past the checks and stops only
    # at the device-memory test of the pointer conversion
    with pytest.raises(ValueError, match="device memory"):
        h = type("H", (), {"handle": None})()
        acpp.inclusive_scan(h, h, t(10), t(10))


def test_group_release_waits_for_plans():
    # bookkeeping only: a group with live plans defers its release
    g = acpp.AllocationGroup.__new__(acpp.AllocationGroup)
    g._h = None
    g._plans = 1
    g._close_pending = False
    g.close()
    assert g._close_pending
    p = acpp.SegmentedPlan.__new__(acpp.SegmentedPlan)
    p._h = None
    p._keep = ()
    p._scratch = g
    p.close()
    assert g._plans == 0
    np.testing.assert_equal(p._scratch, None)


def test_release_refused_while_a_plan_is_alive():
    # a captured graph keeps using the group's regions: releasing them to the
    # cache before the plan is closed would hand them to other calls
    g = acpp.AllocationGroup.__new__(acpp.AllocationGroup)
    g._h = None
    g._plans = 1
    g._close_pending = False
    with pytest.raises(RuntimeError, match="SegmentedPlan"):
        g.release()
    g.close()  # deferred while the plan lives
    assert g._close_pending


@pytest.mark.parametrize("groups", [1, 16, 20])
def test_closed_groups_are_kept_for_new_ones(groups):
    """A cache keeps the handles of at most 16 closed groups per device, hands
    each to one new group only, and gives them back with a purge or its end."""
    cache = acpp.AllocationCache()
    for _ in range(2):
        opened = [acpp.AllocationGroup(cache) for _ in range(groups)]
        assert len({g.handle.value for g in opened}) == groups
        assert not cache._groups[0]
        for g in opened:
            g.close()
            g.close()  # a second close does nothing
            assert g.handle is None
        assert len({h.value for h in cache._groups[0]}) == len(cache._groups[0]) == min(groups, 16)
    cache.purge()
    assert not cache._groups[0]
    late = acpp.AllocationGroup(cache)
    cache_handles = cache._groups[0]
    acpp.AllocationGroup(cache).close()
    assert len(cache_handles) == 1
    late.close()
    cache.close()
    assert not cache_handles


class _Log:
    """The library with every call's name noted."""

    def __init__(self, lib, names):
        self._lib, self._names = lib, names

    def __getattr__(self, name):
        fn = getattr(self._lib, name)

        def call(*args):
            self._names.append(name)
            return fn(*args)
        return call


@pytest.mark.parametrize("groups", [1, 20])
def test_cache_outlives_its_open_groups(monkeypatch, groups):
    # a group's regions go back to its cache: a cache closed first (or
    # finalised first, as the garbage collector may do with a cycle) is
    # destroyed after its last group
    cache = acpp.AllocationCache()
    acpp.AllocationGroup(cache).close()  # one handle kept for new groups
    opened = [acpp.AllocationGroup(cache) for _ in range(groups)]
    names = []
    lib = algorithms._abi.load()
    monkeypatch.setattr(algorithms._abi, "load", lambda: _Log(lib, names))
    cache.close()
    cache.close()
    assert "acpp_allocation_cache_destroy" not in names
    with pytest.raises(acpp.AcppError):
        acpp.AllocationGroup(cache)
    for g in opened:
        g.close()
    assert names.count("acpp_allocation_group_destroy") == groups
    assert names.count("acpp_allocation_cache_destroy") == 1
    assert names[-1] == "acpp_allocation_cache_destroy"
    called = len(names)
    cache.close()
    assert len(names) == called


def test_purge_beside_a_thread_that_takes_the_last_handle():
    class Taken(list):  # not empty when looked at, empty when popped from
        def __len__(self):
            return 1

    cache = acpp.AllocationCache()
    cache._groups[0] = Taken()
    cache.purge()
    cache._groups[0] = []
    cache.close()


def test_last_groups_closed_by_two_threads_destroy_the_cache_once(monkeypatch):
    class Raced(dict):  # another thread is through between a look at it and what follows
        def __len__(self):
            if not self.seen:
                self.seen = True
                cache._destroy()
            return 0

    cache = acpp.AllocationCache()
    names = []
    lib = algorithms._abi.load()
    monkeypatch.setattr(algorithms._abi, "load", lambda: _Log(lib, names))
    cache._alive = Raced()
    cache._alive.seen = False
    cache.close()
    assert names.count("acpp_allocation_cache_destroy") == 1
