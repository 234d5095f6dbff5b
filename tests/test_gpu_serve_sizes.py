"""Queries around the sizes at which their path changes: hits sorted on the
device up to 8192 a hop and by the host beyond, seeds passed in the slot's
page up to 16384 and copied beyond, slots with a page (the first 64) and
without, hit buffers too small for the hits (the query runs again).

A crowd of 1025 objects stands in one spot for ticks 0..6 and is scattered at
tick 7, so every pair of it has met from 0 to 6: a seed of the crowd has 1024
hits, and eight seeds exactly 8192."""
import numpy as np
import pytest

from glint_pipeline_amd import runtime

pytestmark = pytest.mark.gpu

CROWD, N, SIDE, LAST = 1025, 18_000, 20_000.0, 9


@pytest.fixture(scope="module")
def bench():
    rng = np.random.default_rng(5)
    g = np.stack(np.meshgrid(np.arange(140), np.arange(140)), axis=-1).reshape(-1, 2)[:N] * 100.0 + 50.0
    apart = g.astype(np.float64)
    cfg = runtime.make_config(N, (0.0, 0.0, SIDE, SIDE), grid_capacity=64, min_meet_time=3,
                              meeting_log_capacity=1 << 21, contact_capacity=1 << 21)
    wb = runtime.Workbench(cfg)
    made = []

    def server(max_running=4, min_hits=0, index=4, estimate=100):
        sv = runtime.Server(wb, arena_bytes=8 << 30, max_running=max_running, min_hits=min_hits,
                            index_block_ticks=index, estimate_percent=estimate)
        made.append(sv)
        return sv

    first = server()
    bufs = []
    for t in range(LAST + 1):
        xy = apart.copy()
        if t <= 6:
            xy[:CROWD] = rng.uniform(0.0, 0.9, (CROWD, 2)) + 5000.0
        b = runtime.DeviceBuffer(16 * N)
        b.upload(xy)
        bufs.append(b)
        first.tick(t, d_full_xy=b.address())
    wb.synchronize()
    assert wb.meeting_log_info()[0] == CROWD * (CROWD - 1) // 2
    yield wb, first
    for sv in made:
        sv.close()
    wb.close()
    for b in bufs:
        b.free()


def expected(seeds, hops):
    crowd = np.arange(CROWD)
    s = np.array(sorted(v for v in set(seeds) if v < CROWD), dtype=np.int64)

    def rows(sources):
        return np.array([(a, b, 0, 6) for a in sources for b in crowd if a != b], dtype=np.uint32).reshape(-1, 4)

    # every contact's first exposure is at 0, so all of its meetings count
    contacts = np.setdiff1d(crowd, s) if len(s) else s
    return rows(s), rows(contacts) if hops == 2 else rows([])


@pytest.mark.parametrize("hops", [1, 2])
@pytest.mark.parametrize("k", [0, 1, 7, 8, 9])
def test_hits_around_the_device_sort(bench, k, hops):
    _, sv = bench
    seeds = np.concatenate([np.arange(k) * 100, [CROWD + 7]])
    print(f"[serve sizes] {k} seeds of the crowd, {hops} hops", flush=True)
    q = sv.submit(seeds, 0, LAST, hops)
    sv.drain()
    h1, h2 = sv.result(q)
    w1, w2 = expected(seeds, hops)
    assert np.array_equal(h1, w1) and np.array_equal(h2, w2)


@pytest.mark.parametrize("hops", [1, 2])
@pytest.mark.parametrize("nseeds", [16_383, 16_384, 16_385])
def test_seeds_around_the_page(bench, nseeds, hops):
    _, sv = bench
    seeds = np.concatenate([[3, 1000], np.arange(CROWD, CROWD + nseeds - 2)])
    print(f"[serve sizes] {nseeds} seeds, {hops} hops", flush=True)
    q = sv.submit(seeds, 0, LAST, hops)
    sv.drain()
    h1, h2 = sv.result(q)
    w1, w2 = expected(seeds, hops)
    assert np.array_equal(h1, w1) and np.array_equal(h2, w2)
