"""Ticks in which hundreds to thousands of leaves split and merge at once,
around the 512 that one workgroup does alone: leaves, contacts and meetings
equal the oracle's tick by tick and over runs (several contexts together too),
a pool too small for the splits is reported, and the update's time does not
grow with every change."""
import numpy as np
import pytest

from glint_pipeline_amd import gen, runtime
from tests.parity import run_parity

pytestmark = pytest.mark.gpu

CAP = 50


def scene(cells, up, down, ticks, seed=4):
    """cells^2 leaves of 64 m with 13 objects each (four hold more than a leaf may); on even ticks 50 more stand
    in each of `up` of them, on odd ticks in each of `down` others (the rest of
    them over the other leaves): up to `up` splits and `down` merges one tick,
    the reverse the next."""
    rng = np.random.default_rng(seed)
    n = cells * cells
    iy, ix = np.divmod(rng.permutation(n), cells)

    def inside(which):
        return (np.stack([ix, iy], axis=1)[which] + rng.uniform(0.02, 0.98, (len(which), 2))) * 64.0

    loose = inside(np.repeat(np.arange(n), 13))
    movers, others = 50 * max(up, down), np.arange(up + down, n)
    at = []
    for first, count in ((0, up), (up, down)):
        cell = np.concatenate([np.repeat(np.arange(first, first + count), 50),
                               others[np.arange(movers - 50 * count) % len(others)]])
        at.append(np.concatenate([loose, inside(cell)]))
    return [at[t % 2].reshape(-1) for t in range(ticks)], 64.0 * cells


@pytest.mark.parametrize("up,down", [(511, 511), (512, 512), (513, 513), (600, 1), (1, 600), (1500, 1100)])
def test_tick_by_tick(up, down):
    print(f"[schema] {up} up {down} down", flush=True)
    ticks = 6
    pts, side = scene(64, up, down, ticks)
    w = gen.uniform_city(len(pts[0]) // 2, ticks, 500.0, grid_capacity=CAP, min_meet_time=1)   # (its walk is not used)
    run_parity(w, ticks, check_leaves_every=1, box=(0.0, 0.0, side, side), positions=lambda t: pts[t],
               contact_capacity=1 << 20, unit_capacity=1 << 20, node_capacity=1 << 15)


def config(pts, side, **kw):
    kw = {"node_capacity": 1 << 15, "meeting_log_capacity": 1 << 18, **kw}
    return runtime.make_config(len(pts[0]) // 2, (0.0, 0.0, side, side), grid_capacity=CAP, min_meet_time=1,
                               contact_capacity=1 << 20, unit_capacity=1 << 20, **kw)


@pytest.mark.parametrize("graph_ticks", [0, 4])
def test_runs_and_batches(graph_ticks):
    """The same scenes through runs of ticks and in a batch: leaves, meetings
    and active pairs as tick by tick."""
    print(f"[schema] runs and batches, graph_ticks {graph_ticks}", flush=True)
    ticks = 9
    scenes = [scene(64, up, down, ticks, seed) for seed, (up, down) in enumerate([(513, 513), (1500, 1100), (3, 3)])]
    bufs, want = [], []
    for pts, side in scenes:
        with runtime.Workbench(config(pts, side)) as wb:
            for t in range(ticks):
                wb.tick(pts[t], t)
            want.append((wb.leaves(), wb.meeting_log(), wb.active_pairs(), wb.stats()["num_nodes"]))
        bufs.append(runtime.DeviceBuffer(8 * ticks * len(pts[0])))
        bufs[-1].upload(np.concatenate(pts))

    def same(wb, expected):
        leaves, log, active, nodes = expected
        assert all(np.array_equal(a, b) for a, b in zip(wb.leaves(), leaves))
        assert np.array_equal(wb.meeting_log(), log)
        assert all(np.array_equal(a, b) for a, b in zip(wb.active_pairs(), active))
        assert wb.stats()["num_nodes"] == nodes

    for (pts, side), buf, expected in zip(scenes, bufs, want):
        with runtime.Workbench(config(pts, side, graph_ticks=graph_ticks)) as wb:
            wb.run_ticks(buf.address(), 0, ticks)
            same(wb, expected)
    with runtime.Batch([config(*sc) for sc in scenes], graph_ticks=graph_ticks) as bt:
        bt.run_ticks([b.address() for b in bufs], 0, ticks)
        for wb, expected in zip(bt.contexts, want):
            same(wb, expected)
    for b in bufs:
        b.free()


@pytest.mark.parametrize("up", [300, 700])
def test_pool_too_small(up):
    print(f"[schema] {up} splits, too few nodes", flush=True)
    pts, side = scene(32, up, 0, 4)
    with runtime.Workbench(config(pts, side, node_capacity=1365 + 4 * up - 100)) as wb:   # (1365 nodes of the first tree)
        with pytest.raises(runtime.GlintError, match="NODE_CAPACITY"):
            for t in range(4):
                wb.tick(pts[t], t)


def schema_us(up):
    ticks = 8
    pts, side = scene(128, up, up, ticks)
    buf = runtime.DeviceBuffer(8 * ticks * len(pts[0]))
    buf.upload(np.concatenate(pts))
    with runtime.Workbench(config(pts, side, node_capacity=1 << 18)) as wb:
        wb.run_ticks(buf.address(), 0, ticks)
        wb.set_kernel_profiling(True)
        wb.kernel_times(reset=True)
        for rep in range(1, 5):
            wb.run_ticks(buf.address(), rep * ticks, ticks, latencies=False)
        ms, launches = wb.kernel_times()["k_schema"]
        stats = wb.stats()
    assert stats["splits"] == up and stats["merges"] == up
    buf.free()
    return 1e3 * ms / launches


def test_time_of_many_changes():
    """8000 splits and 8000 merges a tick take less than ten times what 10 of
    each take (36 and 7 us; one workgroup alone took 224 and 9)."""
    few, many = schema_us(10), schema_us(8000)
    print(f"[schema] 10 changes {few:.1f} us, 8000 {many:.1f} us", flush=True)
    assert many < 10.0 * few
