"""Queries where their path changes: more running at once than there are slots
with a page (64), hit buffers too small for the first or the second hop (the
query runs again), and more index blocks than a page lists (1024).  The hits
are those of the meeting log, searched on the host."""
import numpy as np
import pytest

from glint_pipeline_amd import runtime

pytestmark = pytest.mark.gpu

GROUP = 24   # objects that meet; 3 GROUP more stand apart


def positions(t, last):
    """Object i of the group stands with i ^ 1 or with i ^ 2 for four ticks in
    turn, each four objects one tick later than the four before."""
    i = np.arange(4 * GROUP)
    xy = np.stack([50.0 * (i % 16) + 25.0, 50.0 * (i // 16) + 25.0], axis=1)
    k = np.arange(GROUP)
    phase = ((t + k // 4) // 4) % 4
    with_ = np.where(phase == 0, k & ~1, np.where(phase == 2, k & ~2, k))
    if t < last - 5:   # the last ticks apart: no pair is in progress
        xy[:GROUP] = xy[with_] + 0.1 * (k & 3)[:, None]
    return xy


def served(wb, sv, ticks, bufs):
    for t in range(ticks):
        b = runtime.DeviceBuffer(16 * 4 * GROUP)
        b.upload(np.ascontiguousarray(positions(t, ticks)))
        bufs.append(b)
        sv.tick(t, d_full_xy=b.address())
    wb.synchronize()
    log = wb.meeting_log().astype(np.int64)
    assert len(log) > ticks // 2
    return log


def expected(log, seeds, hops):
    def rows(start_of):
        out = [(a, b, s, e) for p, q, s, e in log for a, b in ((p, q), (q, p)) if a in start_of and e >= start_of[a]]
        return np.array(sorted(out), dtype=np.uint32).reshape(-1, 4)

    h1 = rows({s: 0 for s in seeds})
    first = {}
    for _, target, start, _ in h1.tolist():
        if target not in seeds:
            first[target] = min(first.get(target, start), start)
    return h1, rows(first) if hops == 2 else rows({})


def config(**kw):
    return runtime.make_config(4 * GROUP, (0.0, 0.0, 800.0, 400.0), grid_capacity=16, min_meet_time=1,
                               meeting_log_capacity=1 << 16, **kw)


def check(sv, log, q, seeds, hops):
    h1, h2 = sv.result(q)
    w1, w2 = expected(log, seeds, hops)
    assert np.array_equal(h1, w1) and np.array_equal(h2, w2), (seeds, hops, len(h1), len(w1), len(h2), len(w2))
    return len(w1), len(w2)


@pytest.mark.parametrize("max_running", [63, 64, 65, 100])
def test_more_queries_than_pages(max_running):
    print(f"[serve slots] {max_running} slots", flush=True)
    ticks, bufs = 60, []
    with runtime.Workbench(config()) as wb, \
            runtime.Server(wb, arena_bytes=1 << 30, max_running=max_running, index_block_ticks=8) as sv:
        log = served(wb, sv, ticks, bufs)
        asked = [([k % GROUP, (k * 7 + 3) % GROUP, GROUP + k % 9], 1 + k % 2) for k in range(150)]
        ids = [sv.submit(seeds, 0, ticks - 1, hops) for seeds, hops in asked]   # (nothing is polled meanwhile)
        running, pending = sv.poll()
        sv.drain()
        total = [check(sv, log, q, set(seeds), hops) for q, (seeds, hops) in zip(ids, asked)]
        assert all(a > 0 for a, _ in total) and sum(b for _, b in total) > 0
    for b in bufs:
        b.free()


@pytest.mark.parametrize("hops", [1, 2])
@pytest.mark.parametrize("index", [8, 0xFFFFFFFF])
def test_buffers_too_small(index, hops):
    """One hit a buffer at first: the first hop's hits do not fit, then the
    second's (more than the first's and one); every query runs again for each."""
    print(f"[serve slots] small buffers, index {index}, {hops} hops", flush=True)
    ticks, bufs = 200, []
    with runtime.Workbench(config()) as wb, \
            runtime.Server(wb, arena_bytes=1 << 28, min_hits=1, estimate_percent=1, index_block_ticks=index) as sv:
        log = served(wb, sv, ticks, bufs)
        retries = []
        for seeds in ([0], [5, 6], [GROUP + 1], [2, 9, 14]):
            q = sv.submit(seeds, 0, ticks - 1, hops)
            sv.drain()
            retries.append(sv.info(q)["retries"])
            n1, n2 = check(sv, log, q, set(seeds), hops)
            assert retries[-1] >= (n1 > 1) + (hops == 2 and n2 > n1 + 1)
        assert max(retries) >= hops
    for b in bufs:
        b.free()


@pytest.mark.parametrize("ticks", [1300, 1450])   # (three ticks of four end a meeting)
def test_more_blocks_than_a_page(ticks):
    print(f"[serve slots] {ticks} ticks, a block each", flush=True)
    bufs = []
    with runtime.Workbench(config()) as wb, runtime.Server(wb, arena_bytes=1 << 28, index_block_ticks=1) as sv:
        log = served(wb, sv, ticks, bufs)
        blocks = sv.index_info()["blocks"]
        assert (blocks > 1024) == (ticks == 1450), blocks
        for seeds, hops in (([3], 1), ([3, 8], 2), ([1, 2, 13], 2)):
            q = sv.submit(seeds, 0, ticks - 1, hops)
            sv.drain()
            check(sv, log, q, set(seeds), hops)
    for b in bufs:
        b.free()
