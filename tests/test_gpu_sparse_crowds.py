"""Crowds in leaves that are sparse on average, which the join hands over from
a wave to the tiles: contacts, meetings, tested pairs and active pairs equal
the oracle's on both sides of every bound (the pairs that a wave's LDS holds,
304 to 368; those it decides, 600, or 1500 with more than 256 sparse leaves;
objects of a cell, 128; columns tested, 1024), beside leaves that stay sparse,
and a crowd takes no longer in a wide leaf than in a narrow one."""
import numpy as np
import pytest

from glint_pipeline_amd import gen, runtime
from tests.parity import run_parity

pytestmark = pytest.mark.gpu

FP64, GUARD = runtime.PRECISION_FP64, runtime.PRECISION_FP32_GUARD


def walk(base, side, ticks, step=0.3, seed=1):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(ticks):
        out.append(np.clip(base, 0.0, side).reshape(-1))
        base = base + rng.uniform(-step, step, base.shape)
    return out


def check(base, side, cap, *, ticks=5, record=True, **kw):
    pts = walk(base, side, ticks)
    w = gen.uniform_city(len(base), ticks, 500.0, grid_capacity=cap, min_meet_time=1)   # (its walk is not used)
    return run_parity(w, ticks, check_contacts=record, box=(0.0, 0.0, side, side), positions=lambda t: pts[t],
                      contact_capacity=1 << 20, unit_capacity=1 << 18, **kw)


def spot(rng, at, k, r=0.3):
    return np.asarray(at) + rng.uniform(-r, r, (k, 2))


@pytest.mark.parametrize("precision,record,complete,tile", [(FP64, True, False, 0), (GUARD, False, False, 0),
                                                            (GUARD, True, True, 512)])
@pytest.mark.parametrize("crowd", [20, 24, 26, 27, 28, 34, 35, 36, 100, 128, 129, 400])
def test_one_spot_in_a_wide_leaf(crowd, precision, record, complete, tile):
    print(f"[crowds] spot of {crowd}, precision {precision} record {record} complete {complete} tile {tile}", flush=True)
    rng = np.random.default_rng(crowd)
    base = np.concatenate([spot(rng, (300.0, 700.0), crowd), rng.uniform(0.0, 1000.0, (30, 2))])
    check(base, 1000.0, 600, precision=precision, record=record, complete=complete, join_tile=tile)


@pytest.mark.parametrize("k,at", [(100, 520.0), (230, 520.0), (420, 520.0), (420, 450.0)])
def test_a_patch_of_a_wide_leaf(k, at):
    """Objects a few reaches apart over 100 m: few pairs, many columns (at 450
    the patch lies over four cells, whose columns add up)."""
    print(f"[crowds] patch of {k} at {at}", flush=True)
    rng = np.random.default_rng(k)
    check(rng.uniform(at, at + 100.0, (k, 2)), 2000.0, 600)


@pytest.mark.parametrize("complete", [False, True])
@pytest.mark.parametrize("few", [1, 12, 70])
def test_units_of_a_crowd_beside_the_leaf(few, complete):
    """480 objects left of a leaf's boundary, within reach of `few` right of it."""
    print(f"[crowds] units, {few} beside, complete {complete}", flush=True)
    rng = np.random.default_rng(few)
    base = np.concatenate([np.stack([rng.uniform(498.6, 499.9, 480), rng.uniform(249.0, 251.0, 480)], axis=1),
                           np.stack([rng.uniform(500.1, 500.5, few), rng.uniform(249.0, 251.0, few)], axis=1),
                           rng.uniform(0.0, 1000.0, (20, 2))])
    check(base, 1000.0, 500, complete=complete)


def many(per, leaves, seed=3):
    """A grid of leaves of 12 objects and a spot of `per`: alternately 0 and
    `per` objects, in 64 m cells of the tree."""
    rng = np.random.default_rng(seed)
    side = 64.0 * leaves
    iy, ix = np.divmod(np.arange(leaves * leaves), leaves)
    loose = (np.repeat(np.stack([ix, iy], axis=1), 12, axis=0) + rng.uniform(0.0, 1.0, (12 * leaves * leaves, 2))) * 64.0
    spots = [spot(rng, (64.0 * x + 32.0, 64.0 * y + 20.0), per) for x, y in zip(ix, iy) if (x + y) % 2]
    return np.concatenate([loose] + spots), side


@pytest.mark.parametrize("precision,record", [(FP64, True), (GUARD, False)])
@pytest.mark.parametrize("per,leaves", [(20, 8), (40, 8), (20, 16), (40, 16), (20, 32), (27, 32), (54, 32), (56, 32),
                                        (90, 32)])
def test_many_leaves(per, leaves, precision, record):
    print(f"[crowds] {leaves}^2 leaves, spots of {per}, precision {precision} record {record}", flush=True)
    base, side = many(per, leaves)
    check(base, side, 110, ticks=3, precision=precision, record=record)


@pytest.mark.parametrize("lat0", [-41.0, 70.0])
def test_lonlat(lat0):
    print(f"[crowds] lon/lat at {lat0}", flush=True)
    proj = runtime.projection_for_box(10.0, lat0)
    fx, fy = proj.deg_per_m_lon, proj.deg_per_m_lat
    for base, side, cap in [(*many(60, 20), 110), (many(100, 4)[0], 256.0, 300)]:
        ticks = 3
        deg = [np.stack([10.0 + p.reshape(-1, 2)[:, 0] * fx, lat0 + p.reshape(-1, 2)[:, 1] * fy], axis=1).reshape(-1)
               for p in walk(base, side, ticks)]
        w = gen.uniform_city(len(base), ticks, 500.0, grid_capacity=cap, min_meet_time=1)   # (its walk is not used)
        run_parity(w, ticks, geography=True, box=(10.0 - fx, lat0 - fy, 10.0 + (side + 1) * fx, lat0 + (side + 1) * fy),
                   positions=lambda t: deg[t], contact_capacity=1 << 20, unit_capacity=1 << 18)


@pytest.mark.parametrize("graph_ticks", [0, 4])
def test_in_a_batch(graph_ticks):
    """Scenes with few and many leaves, with and without crowds, ticked
    together: the same meetings as each alone."""
    print(f"[crowds] batch, graph_ticks {graph_ticks}", flush=True)
    ticks, rng = 9, np.random.default_rng(7)
    one = np.concatenate([spot(rng, (300.0, 700.0), 300), rng.uniform(0.0, 1000.0, (30, 2))])
    scenes = [(one, 1000.0, 600), (*many(56, 24), 110), (rng.uniform(0.0, 4000.0, (9000, 2)), 4000.0, 60),
              (*many(100, 6), 200)]
    cfgs, bufs, want = [], [], []
    for base, side, cap in scenes:
        trace = np.concatenate(walk(base, side, ticks, step=0.8))
        cfgs.append(runtime.make_config(len(base), (0.0, 0.0, side, side), grid_capacity=cap, min_meet_time=1,
                                        meeting_log_capacity=1 << 20, contact_capacity=1 << 20))
        bufs.append(runtime.DeviceBuffer(trace.nbytes))
        bufs[-1].upload(trace)
        with runtime.Workbench(cfgs[-1]) as wb:
            wb.run_ticks(bufs[-1].address(), 0, ticks)
            want.append((wb.meeting_log(), wb.active_pairs()))
    with runtime.Batch(cfgs, graph_ticks=graph_ticks) as bt:
        bt.run_ticks([b.address() for b in bufs], 0, ticks)
        for i, (log, active) in enumerate(want):
            assert len(log) > 0
            assert np.array_equal(bt.contexts[i].meeting_log(), log), f"scene {i}: meetings"
            assert all(np.array_equal(a, b) for a, b in zip(bt.contexts[i].active_pairs(), active)), f"scene {i}"
    for b in bufs:
        b.free()


def tick_ms(base, side, cap, complete=False):
    ticks = 8
    trace = np.concatenate(walk(base, side, ticks, step=0.02))
    buf = runtime.DeviceBuffer(trace.nbytes)
    buf.upload(trace)
    ms = []
    with runtime.Workbench(runtime.make_config(len(base), (0.0, 0.0, side, side), grid_capacity=cap, complete=complete,
                                               contact_capacity=1 << 21, unit_capacity=1 << 18)) as wb:
        for rep in range(6):
            m = wb.run_ticks(buf.address(), rep * ticks, ticks)
            ms += m[1:].tolist() if rep else []
    buf.free()
    return float(np.median(ms))


def test_a_crowd_is_no_slower_in_a_wide_leaf():
    """The same objects in a box 40 m and a kilometre wide, where a leaf is
    dense and sparse: within a factor of two (they differ by 2 to 10 %; a wave
    alone takes four times as long, and six for a crowd's units)."""
    rng = np.random.default_rng(4)
    for k in (160, 320, 480):
        crowd = spot(rng, (20.0, 20.0), k)
        narrow, wide = tick_ms(crowd, 40.0, 600), tick_ms(crowd, 1000.0, 600)
        print(f"[crowds] {k} in one spot: {1e3 * narrow:.0f} us in 40 m, {1e3 * wide:.0f} in 1000 m", flush=True)
        assert wide < 2.0 * narrow
    # the crowd beside 12 objects of another leaf: the wide leaf's units
    def beside(side):
        m = side / 2
        return np.concatenate([np.stack([rng.uniform(m - 1.4, m - 0.1, 480), rng.uniform(m / 2 - 1, m / 2 + 1, 480)], axis=1),
                               np.stack([rng.uniform(m + 0.1, m + 0.5, 12), rng.uniform(m / 2 - 1, m / 2 + 1, 12)], axis=1)])
    narrow, wide = tick_ms(beside(16.0), 16.0, 485, True), tick_ms(beside(1000.0), 1000.0, 485, True)
    print(f"[crowds] units: {1e3 * narrow:.0f} us in 16 m, {1e3 * wide:.0f} in 1000 m", flush=True)
    assert wide < 2.0 * narrow
