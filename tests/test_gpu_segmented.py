"""GPU parity: segmented inclusive scans and reductions, direct and through
hipGraph plans, against the oracle's per-segment serial scan / fold."""
import math

import numpy as np
import pytest

import opensycl_amd as acpp
import oracle as O
from gpu_util import dev, exact_ints, fold_bound, host, lognormal_offsets, rand, scan_depth

# segmented tiles hold at least 128 work-items x 2 rows x 16 bytes
MIN_TILE = 512

pytestmark = pytest.mark.gpu


def layouts():
    rng = np.random.default_rng(5)
    yield "lognormal", lognormal_offsets(3000, seed=1, max_len=1 << 18)
    yield "ones", np.arange(0, 20001, dtype=np.uint64)
    lens = rng.integers(0, 5, 5000).astype(np.uint64)  # many empty segments
    yield "with_empty", np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    yield "one_huge", np.array([0, (1 << 22) + 77], dtype=np.uint64)
    lens = np.array([0, 0, 3, 0, 70000, 0, 1, 123456, 0], dtype=np.uint64)
    yield "mixed_edges", np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)


def _values(dtype, n, seed):
    if np.issubdtype(dtype, np.floating):
        return rand(dtype, n, seed)
    return rand(dtype, n, seed, lo=-(1 << 20), hi=1 << 20)


@pytest.mark.parametrize("dtype", [np.int32, np.int64, np.float32, np.float64])
def test_segmented_scan(gpu, q, scratch, dtype):
    torch, _ = gpu
    for name, off in layouts():
        n = int(off[-1])
        x = _values(dtype, n, seed=n)
        xd, od = dev(torch, x), dev(torch, off)
        for op in (acpp.PLUS, acpp.MAX):
            yd = torch.zeros_like(xd)
            acpp.segmented_inclusive_scan(q, scratch, xd, yd, od, op)
            q.wait()
            got = host(yd)
            if np.issubdtype(dtype, np.floating) and op == acpp.PLUS:
                # FP64 per-segment prefix sums; fold depth bound per element
                eps = np.finfo(dtype).eps
                ok = True
                x64 = x.astype(np.float64)
                for s in range(len(off) - 1):
                    b, e = int(off[s]), int(off[s + 1])
                    if e > b:
                        ex = np.cumsum(x64[b:e])
                        bound = fold_bound(np.cumsum(np.abs(x64[b:e])),
                                           scan_depth(np.arange(e - b), MIN_TILE), eps)
                        ok &= bool(np.all(np.abs(got[b:e].astype(np.float64) - ex) <= bound + 1e-300))
                assert ok, (name, op)
            else:
                assert np.array_equal(got, O.segmented_inclusive_scan(x, off, op)), (name, op)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_segmented_exact_fp(gpu, q, scratch, dtype):
    # integer-valued floats: per-segment sums and prefix sums are exact, so
    # the floating-point kernels must agree bit for bit with the oracle's
    # integer scan and fold; a lost or duplicated element fails here
    torch, _ = gpu
    tdt = torch.float32 if dtype == np.float32 else torch.float64
    for name, off in layouts():
        n = int(off[-1])
        xi = exact_ints(torch, n, n % 1000)
        xh = host(xi).astype(np.int64)
        xd, od = xi.to(tdt), dev(torch, off)
        yd = torch.zeros_like(xd)
        acpp.segmented_inclusive_scan(q, scratch, xd, yd, od)
        out = torch.zeros(len(off) - 1, dtype=tdt, device="cuda")
        acpp.segmented_reduce(q, scratch, xd, od, out, 0.0)
        q.wait()
        assert np.array_equal(host(yd).astype(np.int64), O.segmented_inclusive_scan(xh, off)), name
        assert np.array_equal(host(out).astype(np.int64), O.segmented_reduce(xh, off, np.int64(0))), name


@pytest.mark.parametrize("dtype", [np.int32, np.int64, np.float32, np.float64])
def test_segmented_reduce(gpu, q, scratch, dtype):
    torch, _ = gpu
    for name, off in layouts():
        n = int(off[-1])
        S = len(off) - 1
        x = _values(dtype, n, seed=n + 1)
        xd, od = dev(torch, x), dev(torch, off)
        for op, init in ((acpp.PLUS, dtype(7)), (acpp.MIN, dtype(1 << 20)), (acpp.MAX, dtype(-5))):
            out = torch.full((S,), -99, dtype=xd.dtype, device="cuda")
            acpp.segmented_reduce(q, scratch, xd, od, out, init, op)
            q.wait()
            got = host(out)
            if np.issubdtype(dtype, np.floating) and op == acpp.PLUS:
                exact = O.segmented_reduce_f32_fp64(x.astype(np.float32), off) if dtype == np.float32 \
                    else np.array([math.fsum(x[int(off[s]):int(off[s + 1])]) for s in range(S)])
                lens = np.diff(off.astype(np.int64))
                absx = np.abs(x.astype(np.float64))
                abs_sums = np.array([absx[int(off[s]):int(off[s + 1])].sum() for s in range(S)])
                eps = np.finfo(dtype).eps
                bound = fold_bound(abs_sums + 7, scan_depth(lens, MIN_TILE) + 1, eps) + 1e-300
                assert np.all(np.abs(got.astype(np.float64) - (exact + 7)) <= bound), name
            else:
                assert np.array_equal(got, O.segmented_reduce(x, off, init, op)), (name, op)


# flags: 1 = work-group-wide look-back window, 4 = one work-group per tile.
# (64, 2) gives 256-element int64 tiles: thousands of single-wave tiles in
# flight, the heaviest look-back contention (a regression case for the
# look-back backoff; without it the look-backs ran out of time).
@pytest.mark.parametrize("cfg", [(64, 2), (128, 4), (256, 2), (512, 4), (1024, 2), (1024, 4),
                                 (256, 4, 0, 1), (256, 4, 0, 4), (512, 8, 0, 5), (64, 2, 0, 4),
                                 (1024, 8, 0, 0), (64, 2, 0, 1)])
def test_segmented_configs(gpu, q, scratch, cfg):
    torch, _ = gpu
    off = lognormal_offsets(2000, seed=3, max_len=1 << 17)
    n = int(off[-1])
    x = rand(np.int64, n, seed=9, lo=-1000, hi=1000)
    xd, od = dev(torch, x), dev(torch, off)
    yd = torch.zeros_like(xd)
    acpp.segmented_inclusive_scan(q, scratch, xd, yd, od, acpp.PLUS, config=cfg)
    out = torch.zeros(len(off) - 1, dtype=torch.int64, device="cuda")
    acpp.segmented_reduce(q, scratch, xd, od, out, np.int64(0), acpp.PLUS, config=cfg)
    q.wait()
    assert scratch.watchdog_trips() == 0
    assert np.array_equal(host(yd), O.segmented_inclusive_scan(x, off))
    assert np.array_equal(host(out), O.segmented_reduce(x, off, np.int64(0)))


def test_segmented_plan_replays(gpu, q, scratch):
    # hipGraph replays, each checked, with eager work between replays
    torch, _ = gpu
    off = lognormal_offsets(4000, seed=4, max_len=1 << 18)
    n = int(off[-1])
    x = rand(np.int64, n, seed=2, lo=-(1 << 20), hi=1 << 20)
    xd, od = dev(torch, x), dev(torch, off)
    yd = torch.zeros_like(xd)
    f = rand(np.float32, n, seed=3)
    fd = dev(torch, f)
    red = torch.zeros(len(off) - 1, dtype=torch.float32, device="cuda")
    scan_plan = acpp.SegmentedPlan.inclusive_scan(scratch, xd, yd, od)
    red_plan = acpp.SegmentedPlan.reduce(scratch, fd, od, red, 0.0)
    exp_scan = O.segmented_inclusive_scan(x, off)
    exact = O.segmented_reduce_f32_fp64(f, off)
    lens = np.diff(off.astype(np.int64))
    abs_sums = O.segmented_reduce_f32_fp64(np.abs(f), off)
    bound = fold_bound(abs_sums, scan_depth(lens, MIN_TILE), np.finfo(np.float32).eps) + 1e-30
    for rep in range(4):
        yd.zero_()
        red.zero_()
        scan_plan.launch(q)
        red_plan.launch(q)
        q.wait()
        assert np.array_equal(host(yd), exp_scan), rep
        got = host(red).astype(np.float64)
        assert np.all(np.abs(got - exact) <= bound), rep
        # eager work on the same stream between replays
        tmp = torch.zeros_like(xd)
        acpp.inclusive_scan(q, scratch, xd, tmp)
        q.wait()
        # change the input: the next replay must see the new values
        x = x + 1
        xd.copy_(dev(torch, x))
        exp_scan = O.segmented_inclusive_scan(x, off)
    scan_plan.close()
    red_plan.close()


def test_segmented_lognormal_workload_shape(gpu, q, scratch):
    # 65,536 segments, log-normal lengths (median 512, sigma 2, clipped to
    # [1, 2^20]): int64 segmented inclusive scan, exact
    torch, _ = gpu
    off = lognormal_offsets(65536, seed=0)
    n = int(off[-1])
    x = rand(np.int64, n, seed=7, lo=-(1 << 20), hi=1 << 20)
    xd, od = dev(torch, x), dev(torch, off)
    yd = torch.empty_like(xd)
    acpp.segmented_inclusive_scan(q, scratch, xd, yd, od)
    q.wait()
    y = host(yd)
    del yd
    assert np.array_equal(y, O.segmented_inclusive_scan(x, off))


def test_segmented_plan_first_capture_allocates(gpu, q):
    # A plan made with a fresh cache has to allocate its scratch while the
    # launch is being captured; the plan must still work, and later torch
    # work must not see a stale HIP error.
    torch, _ = gpu
    off = lognormal_offsets(500, seed=8, max_len=1 << 15)
    n = int(off[-1])
    x = rand(np.int64, n, seed=4, lo=-1000, hi=1000)
    xd, od = dev(torch, x), dev(torch, off)
    yd = torch.zeros_like(xd)
    cache = acpp.AllocationCache()
    with acpp.AllocationGroup(cache, 0) as g:
        plan = acpp.SegmentedPlan.inclusive_scan(g, xd, yd, od)
        plan.launch(q)
        q.wait()
        assert np.array_equal(host(yd), O.segmented_inclusive_scan(x, off))
        z = torch.ones(1000, device="cuda").cumsum(0)  # torch work after the capture
        assert z[-1].item() == 1000.0
        plan.close()
    cache.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_segmented_views_one_element_off(gpu, q, scratch, dtype):
    # input and output views one element into their buffers (not 16-byte
    # aligned): 16-byte accesses at element alignment
    torch, _ = gpu
    off = lognormal_offsets(3000, seed=11, max_len=1 << 16)
    n = int(off[-1])
    x = rand(dtype, n + 1, seed=12, lo=-1000, hi=1000)
    xd = dev(torch, x)[1:]
    od = dev(torch, off)
    yb = torch.zeros(n + 1, dtype=xd.dtype, device="cuda")
    acpp.segmented_inclusive_scan(q, scratch, xd, yb[1:], od, acpp.PLUS)
    out = torch.zeros(len(off) - 1, dtype=xd.dtype, device="cuda")
    acpp.segmented_reduce(q, scratch, xd, od, out, dtype(0), acpp.PLUS)
    q.wait()
    assert np.array_equal(host(yb)[1:], O.segmented_inclusive_scan(x[1:], off))
    assert np.array_equal(host(out), O.segmented_reduce(x[1:], off, dtype(0), acpp.PLUS))


def test_plan_keeps_its_group_and_buffers_alive(gpu, q):
    # A plan built from a temporary group and temporary tensors: after the
    # builder's references are gone and the allocator and cache have been
    # churned, a replay still scans the right data into the right output.
    import gc
    torch, cache = gpu
    off = lognormal_offsets(500, seed=9, max_len=1 << 14)
    n = int(off[-1])
    x = rand(np.int64, n, seed=9, lo=-1000, hi=1000)

    def make():
        g = acpp.AllocationGroup(cache, 0)
        xd, od = dev(torch, x), dev(torch, off)
        yd = torch.zeros_like(xd)
        return acpp.SegmentedPlan.inclusive_scan(g, xd, yd, od), yd

    plan, yd = make()
    gc.collect()
    junk = [torch.full((n,), 7, dtype=torch.int64, device="cuda") for _ in range(3)]
    with acpp.AllocationGroup(cache, 0) as other:
        acpp.inclusive_scan(q, other, junk[0], junk[1])
        plan.launch(q)
        acpp.inclusive_scan(q, other, junk[1], junk[2])
        q.wait()
    assert np.array_equal(host(yd), O.segmented_inclusive_scan(x, off))
    assert int(host(junk[2])[-1]) == 7 * n * (n + 1) // 2  # n < 2^23: no wrap
    plan.close()


def _edge_layouts():
    rng = np.random.default_rng(11)

    def of(lens):
        return np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)

    yield "no_elements", of([0] * 300)
    yield "one_element", of([0, 1, 0])
    # starts on, before and after multiples of every tile size (512 .. 32768)
    yield "tile_edges", of([511, 1, 0, 0, 512, 1023, 1, 2049, 0, 4095, 4096, 0, 8191, 1, 0, 32768, 32767, 0])
    yield "three_and_four_starts", of([600, 700, 800] * 30 + [500, 500, 500, 500] * 30)
    # more than 1024 starts in a tile, with empty segments
    yield "ones_and_empty", of(rng.integers(0, 2, 60000))
    # more than 4096 segments, fewer and more than 16 a tile, over 1024 tiles
    # of the (64, 2) configuration below
    yield "many_long", of(rng.integers(0, 400, 9000))
    yield "many_short", of(rng.integers(0, 9, 400000))
    # one segment over more than 1024 tiles, some over 17 .. 1024 tiles
    yield "spans", of([3, 1 << 20, 0, 20000, 9000, 5, 500000, 77])


# (64, 2): 512 (4-byte) or 256 (8-byte) elements a tile, so the table of the
# tiles' segments and every span of the fix-up; default: the library's tiles
@pytest.mark.parametrize("dtype", [np.int32, np.int64, np.float64])
@pytest.mark.parametrize("cfg", [(64, 2), (1024, 8), None])
def test_segmented_edges(gpu, q, scratch, dtype, cfg):
    torch, _ = gpu
    for name, off in _edge_layouts():
        n = int(off[-1])
        # small integers: sums are exact in any order
        x = _values(np.int32, n, seed=n + 2) % 1000 if n else np.zeros(0, np.int32)
        x = x.astype(dtype)
        xd, od = dev(torch, x), dev(torch, off)
        xi = x.astype(np.int64)
        for op, init in ((acpp.PLUS, 7), (acpp.MAX, -2000)):
            out = torch.full((len(off) - 1,), -99, dtype=xd.dtype, device="cuda")
            acpp.segmented_reduce(q, scratch, xd, od, out, init, op, config=cfg)
            yd = torch.full_like(xd, -99)
            acpp.segmented_inclusive_scan(q, scratch, xd, yd, od, op, config=cfg)
            q.wait()
            scratch.release()
            exp = O.segmented_reduce(xi, off, np.int64(init), op)
            assert np.array_equal(host(out).astype(np.int64), exp), (name, op)
            if n:
                assert np.array_equal(host(yd).astype(np.int64), O.segmented_inclusive_scan(xi, off, op)), (name, op)


@pytest.mark.parametrize("n", [5000, 1 << 21, (1 << 23) + 5])
def test_plan_launched_eagerly_and_in_a_graph(gpu, n):
    # a plan's launches continue its region's epochs, also on another stream
    # and after replays of a graph that holds one
    torch, _ = gpu
    off = np.concatenate([[0], np.sort(np.random.default_rng(n).integers(0, n, 300)), [n]]).astype(np.uint64)
    x = exact_ints(torch, n, 3)
    od = dev(torch, off)
    cache = acpp.AllocationCache()
    scratch = acpp.AllocationGroup(cache)
    yd = torch.zeros_like(x)
    out = torch.zeros(len(off) - 1, dtype=x.dtype, device="cuda")
    scan = acpp.SegmentedPlan.inclusive_scan(scratch, x, yd, od)
    red = acpp.SegmentedPlan.reduce(scratch, x, od, out)

    def check(what):
        torch.cuda.synchronize()
        xh = host(x)
        assert np.array_equal(host(yd), O.segmented_inclusive_scan(xh, off)), what
        assert np.array_equal(host(out), O.segmented_reduce(xh, off, np.int32(0))), what
        yd.zero_()
        out.zero_()
        x.add_(1)

    side = torch.cuda.Stream()
    for what in ("first", "second"):
        scan.launch(acpp.Queue())
        red.launch(acpp.Queue())
        check(what)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        scan.launch(acpp.Queue())
        red.launch(acpp.Queue())
    for what in range(3):
        graph.replay()
        check(("replay", what))
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            scan.launch(acpp.Queue())
            red.launch(acpp.Queue())
        check(("eager after replay", what))
    del graph
    scan.close()
    red.close()
    scratch.close()
    cache.close()


# Large reductions: few segments and one more than few (the tile differs), and
# segments of very different lengths, whose tiles one work-item, 16 lanes or
# the whole group write.
@pytest.mark.parametrize("segments", [1, 5, 95, 96, 768, 769, 4000])
def test_segmented_reduce_tiles_by_segments(gpu, q, scratch, segments):
    torch, _ = gpu
    n = 768 << 14  # 48 MiB of int32
    gen = torch.Generator().manual_seed(segments)
    cuts = (torch.rand(segments - 1, generator=gen).double() ** 3 * n).long().sort().values
    offsets = torch.cat([torch.tensor([0]), cuts, torch.tensor([n])])
    x = torch.randint(-1000, 1000, (n,), dtype=torch.int32, generator=gen)
    sums = torch.cat([torch.tensor([0]), x.long().cumsum(0)])[offsets]
    out = torch.zeros(segments, dtype=torch.int32, device="cuda")
    acpp.segmented_reduce(q, scratch, x.cuda(), offsets.cuda().view(torch.uint64), out)
    q.wait()
    assert torch.equal(out.cpu().long(), sums[1:] - sums[:-1])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("lens", [[1], [1, 1, 1], [3, 70, 1], [200, 1, 900], [5000, 2, 3000], [100000, 50001, 1],
                                  [1 << 22, 77], [9] * 3000], ids=lambda l: f"{len(l)}x{l[0]}")
def test_segmented_min_max_nan_and_infinities(gpu, q, scratch, dtype, lens):
    # A NaN as the last element of every other segment, and infinities.  Whatever
    # the order of its elements, a segment with a NaN gives that NaN or one of
    # the segment's numbers; the others give the exact result.
    torch, _ = gpu
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    n, S = int(off[-1]), len(lens)
    first, last = off[:-1].astype(np.int64), off[1:].astype(np.int64) - 1
    for op, init, worst in ((acpp.MAX, -np.inf, -np.inf), (acpp.MIN, np.inf, np.inf)):
        x = np.round(rand(np.float64, n, seed=S) * 100).astype(dtype)
        x[np.arange(1, n, 1013)] = -worst
        x[first[1::4]] = worst
        x[last[::2]] = np.nan
        out = torch.zeros(S, dtype=torch.float32 if dtype == np.float32 else torch.float64, device="cuda")
        acpp.segmented_reduce(q, scratch, dev(torch, x), dev(torch, off), out, init, op)
        q.wait()
        got = host(out)
        for s in range(S):
            seg = x[first[s]:last[s] + 1]
            if s % 2 == 0:
                assert np.isnan(got[s]) or got[s] in seg, (op, s, got[s])
            else:
                assert got[s] == (seg.max() if op == acpp.MAX else seg.min()), (op, s, got[s])


def _empty_run_layouts():
    """Runs of empty segments from a few to far more than a work-group walks, in
    front, inside a tile, at a tile's edge and behind the last element, and
    segments that are empty nearly everywhere."""
    rng = np.random.default_rng(17)
    for n in (0, 5, 1000, 70001, (1 << 20) + 13, 1 << 20, (1 << 23) + 77):
        lens = np.bincount(rng.integers(0, 40, n), minlength=40) if n else np.zeros(0, dtype=np.int64)
        for run in (300, 16384, 16385, 40000, 200001):
            for at in sorted({0, len(lens) // 2, len(lens)}):
                yield f"{run} at {at} of {n}", np.concatenate([lens[:at], np.zeros(run, dtype=np.int64), lens[at:]])
        if n:
            # runs at single elements, next to each other and at round positions
            pos = np.unique(np.concatenate([[0, 1, 2, 31, 32, 33, 4096, 8191, 8192], rng.integers(0, n, 5), [n - 1, n]]))
            off = np.sort(np.concatenate([np.repeat(pos[pos <= n], 20000), [0, n]]))
            yield f"many runs in {n}", np.diff(off)
            yield f"sparse in {n}", np.bincount(rng.integers(0, 300000, n), minlength=300000)


@pytest.mark.parametrize("dtype", [np.int32, np.float64])
def test_runs_of_empty_segments(gpu, q, scratch, dtype):
    torch, _ = gpu
    for name, lens in _empty_run_layouts():
        off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
        n, S = int(off[-1]), len(lens)
        xi = exact_ints(torch, n, n % 1000)
        xh = host(xi).astype(np.int64)
        xd, od = xi.to(torch.int32 if dtype == np.int32 else torch.float64), dev(torch, off)
        if n:
            yd = torch.zeros_like(xd)
            acpp.segmented_inclusive_scan(q, scratch, xd, yd, od)
            q.wait()
            assert np.array_equal(host(yd).astype(np.int64), O.segmented_inclusive_scan(xh, off)), name
        out = torch.full((S,), -7, dtype=xd.dtype, device="cuda")
        acpp.segmented_reduce(q, scratch, xd, od, out, 3)
        q.wait()
        assert np.array_equal(host(out).astype(np.int64), O.segmented_reduce(xh, off, np.int64(3))), name
        scratch.release()


@pytest.mark.parametrize("cfg", [(64, 2), (128, 8), (1024, 2), (1024, 8)])
def test_runs_of_empty_segments_tile_sizes(gpu, q, scratch, cfg):
    # the same with every tile size from the smallest to the largest
    torch, _ = gpu
    n = 300007
    rng = np.random.default_rng(23)
    pos = np.concatenate([np.repeat([0, 511, 512, 32767, 32768, 150000, n], 40000), rng.integers(0, n, 30000), [0, n]])
    off = np.sort(pos).astype(np.uint64)
    xi = exact_ints(torch, n, 1)
    xh = host(xi).astype(np.int64)
    config = {"work_group_size": cfg[0], "items_per_thread": cfg[1]}
    yd = torch.zeros_like(xi)
    out = torch.full((len(off) - 1,), -7, dtype=xi.dtype, device="cuda")
    acpp.segmented_inclusive_scan(q, scratch, xi, yd, dev(torch, off), config=config)
    acpp.segmented_reduce(q, scratch, xi, dev(torch, off), out, 3, config=config)
    q.wait()
    assert np.array_equal(host(yd).astype(np.int64), O.segmented_inclusive_scan(xh, off))
    assert np.array_equal(host(out).astype(np.int64), O.segmented_reduce(xh, off, np.int64(3)))


@pytest.mark.parametrize("starts", [[40], [0, 63], [1, 31, 32], [0, 1, 33, 63], [2, 3, 31, 32, 62], list(range(64))])
def test_runs_of_empty_segments_in_one_block(gpu, q, scratch, starts):
    # as many distinct starts as are found one after the other, and more, in 64
    # elements: at the input's front, inside a tile, and in front of its end
    torch, _ = gpu
    for n in (64, 5000, 70016, 1 << 20):
        for block in sorted({0, (n // 3) & ~63, n - 64}):
            for spare in ([], np.arange(0, n, 3)):
                pos = np.concatenate([np.repeat(block + np.array(starts), 20000), spare, [0, n]])
                off = np.sort(pos).astype(np.uint64)
                xi = exact_ints(torch, n, block)
                xh = host(xi).astype(np.int64)
                yd = torch.zeros_like(xi)
                out = torch.full((len(off) - 1,), -7, dtype=xi.dtype, device="cuda")
                acpp.segmented_inclusive_scan(q, scratch, xi, yd, dev(torch, off))
                acpp.segmented_reduce(q, scratch, xi, dev(torch, off), out, 3)
                q.wait()
                assert np.array_equal(host(yd).astype(np.int64), O.segmented_inclusive_scan(xh, off)), (n, block)
                assert np.array_equal(host(out).astype(np.int64), O.segmented_reduce(xh, off, np.int64(3))), (n, block)
                scratch.release()


@pytest.mark.parametrize("kind", ["scan", "reduce"])
@pytest.mark.parametrize("n", [1 << 20, 1 << 23])
def test_runs_of_empty_segments_cost_what_spread_ones_cost(gpu, q, scratch, kind, n):
    # 4 million empty segments in one place against as many spread over the
    # input: one work-group that walks the run alone takes 50 times as long
    torch, _ = gpu
    S = 4_000_000
    spread = np.sort(np.random.default_rng(1).integers(0, n, S + 1))
    spread[0], spread[-1] = 0, n
    one = np.concatenate([np.linspace(0, n // 2, 500), np.full(S - 999, n // 2), np.linspace(n // 2, n, 500)])
    x = torch.ones(n, dtype=torch.int32, device="cuda")
    d = torch.empty(n if kind == "scan" else S, dtype=torch.int32, device="cuda")
    times = []
    for off in (spread, one):
        od = dev(torch, off.astype(np.uint64))
        assert od.numel() == S + 1
        samples = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            if kind == "scan":
                acpp.segmented_inclusive_scan(q, scratch, x, d, od)
            else:
                acpp.segmented_reduce(q, scratch, x, od, d, 0)
            b.record()
            b.synchronize()
            scratch.release()
            samples.append(a.elapsed_time(b))
        times.append(min(samples))
    assert times[1] < 5 * times[0], times


@pytest.mark.parametrize("wg", [64, 128, 192, 512, 960, 1024])
@pytest.mark.parametrize("n", [(1 << 20) - 1, 1 << 20, 4_000_001])
def test_segmented_scan_with_a_width_alone(gpu, q, scratch, wg, n):
    # the rows then follow the width: the default tile's size, up to 8 rows
    torch, _ = gpu
    rng = np.random.default_rng(wg)
    off = np.concatenate([[0], np.sort(rng.integers(0, n, 3000)), [n]]).astype(np.uint64)
    xi = exact_ints(torch, n, wg)
    xh = host(xi).astype(np.int64)
    for dt in (torch.int32, torch.float64):
        yd = torch.zeros(n, dtype=dt, device="cuda")
        acpp.segmented_inclusive_scan(q, scratch, xi.to(dt), yd, dev(torch, off), config={"work_group_size": wg})
        q.wait()
        assert np.array_equal(host(yd).astype(np.int64), O.segmented_inclusive_scan(xh, off)), dt
