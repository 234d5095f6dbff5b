"""The number of contacts asked for alone equals the list's and the oracle's
between the stages of a tick, before evaluation (from the list) as after it
(from the counters), in planar metres and in lon/lat degrees, where a pair
found from both sides may pass the test from one only."""
import ctypes

import numpy as np
import pytest

from glint_pipeline_amd import gen, runtime
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def counts(wb):
    n, m = ctypes.c_uint64(), ctypes.c_uint64()
    wb._chk(runtime.lib().glint_contacts(wb.h, None, 0, ctypes.byref(n)), "glint_contacts")
    out = np.zeros(1 << 16, dtype=np.uint64)
    wb._chk(runtime.lib().glint_contacts(wb.h, out.ctypes.data, out.size, ctypes.byref(m)), "glint_contacts")
    return n.value, m.value


@pytest.mark.parametrize("complete", [False, True])
@pytest.mark.parametrize("lat", [None, -41.0, 75.0])
@pytest.mark.parametrize("cap", [4, 40])
def test_count_between_stages(cap, lat, complete):
    print(f"[contacts stages] cap {cap} lat {lat} complete {complete}", flush=True)
    n, side = 3000, 250.0
    w = gen.uniform_city(n, 6, side, grid_capacity=cap, seed=4)
    g = gen.Generator(w)
    box, place = w.box(), (lambda xy: xy)
    if lat is not None:
        p = runtime.projection_for_box(10.0, lat)
        box = (10.0 - p.deg_per_m_lon, lat - p.deg_per_m_lat, 10.0 + (side + 1) * p.deg_per_m_lon,
               lat + (side + 1) * p.deg_per_m_lat)
        place = lambda xy: np.stack([10.0 + xy.reshape(-1, 2)[:, 0] * p.deg_per_m_lon,   # noqa: E731
                                     lat + xy.reshape(-1, 2)[:, 1] * p.deg_per_m_lat], axis=1).reshape(-1)
    geo = lat is not None
    o = Oracle(n, box, w.reach_distance, cap, w.min_meet_time, complete=complete, geography=geo)
    cfg = runtime.make_config(n, box, grid_capacity=cap, record_contacts=True, complete=complete, geography=geo,
                              contact_capacity=1 << 17, unit_capacity=1 << 18)
    with runtime.Workbench(cfg) as wb:
        for t in range(5):
            xy = place(g.positions() if t == 0 else g.step())
            o.tick(xy, t)
            want = len(o.contacts())
            assert want > 100
            wb.set_points(xy, t)
            wb.filter()
            wb.reachability()
            assert counts(wb) == (want, want)
            wb.update_meetings()
            assert counts(wb) == (want, want)
            wb.update_schema()
            assert counts(wb) == (want, want)
    o.close()
