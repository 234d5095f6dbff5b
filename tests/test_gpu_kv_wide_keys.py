"""Key-value flushes whose keys differ in more or fewer bits than a 64-bit
sort key holds: ticks far apart make durations and ends differ in up to 23
bits each beside the ids' 24, ticks one apart in a handful.  Every part of
every flush equals the oracle's, bit for bit.  (Contacts are recorded, which
keeps every pair in the table: a pair that ends after a single tick is only
ever emitted when ticks are far apart.)"""
import numpy as np
import pytest

from glint_pipeline_amd import gen, runtime
from oracle.oracle import Oracle
from tests.test_gpu_kv import assert_flush_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("step", [1, 1 << 4, 1 << 10, 1 << 14, 1 << 17])
@pytest.mark.parametrize("area", [1e9, 600.0])
def test_flushes_with_spread_ticks(step, area):
    rng = np.random.default_rng(step)
    w = gen.uniform_city(2500, 60, 500.0, seed=5, grid_capacity=16, min_meet_time=3)
    g = gen.Generator(w)
    o = Oracle(w.num_objects, w.box(), w.reach_distance, w.grid_capacity, w.min_meet_time)
    limit = 64 * step + 8
    o.kv_enable(split_num=4, max_meet_time=limit, area_limit=area)
    cfg = runtime.make_config(w.num_objects, w.box(), reach_distance=w.reach_distance, grid_capacity=w.grid_capacity,
                              min_meet_time=w.min_meet_time, max_meet_time=limit, kv_capacity=1 << 16, kv_split_num=4,
                              kv_area_limit=area, record_contacts=True)
    print(f"[kv wide] step {step} area {area}", flush=True)
    t, keys = 0, 0
    with runtime.Workbench(cfg) as wb:
        for k in range(60):
            xy = (g.positions() if k == 0 else g.step()).copy()
            o.tick(xy, t)
            assert np.array_equal(wb.tick(xy, t), o.meetings()), f"tick {t}"
            if k in (30, 59):
                got, want = wb.kv_flush(), o.kv_flush()
                assert_flush_equal(got, want, f"tick {t}")
                keys += want["summary"]["kept_keys"] + want["summary"]["oversize_keys"]
            t += int(rng.integers(1, step + 1))
    o.close()
    assert keys > 1000
