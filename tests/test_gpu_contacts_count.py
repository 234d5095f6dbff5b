"""The number of contacts that a caller asks for first equals the number that
the list then has, and the oracle's: after stage calls (before and after
evaluation), runs of ticks, and in a restored context; with many pairs found
twice (small leaves), none, lon/lat degrees, and no pairs at all."""
import ctypes

import numpy as np
import pytest

from glint_pipeline_amd import gen, runtime
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def counts(wb):
    """The number alone, and the number with the list."""
    n, m = ctypes.c_uint64(), ctypes.c_uint64()
    wb._chk(runtime.lib().glint_contacts(wb.h, None, 0, ctypes.byref(n)), "glint_contacts")
    out = np.zeros(1 << 16, dtype=np.uint64)
    wb._chk(runtime.lib().glint_contacts(wb.h, out.ctypes.data, out.size, ctypes.byref(m)), "glint_contacts")
    return n.value, m.value


@pytest.mark.parametrize("complete", [False, True])
@pytest.mark.parametrize("n,side,cap", [(2, 500.0, 4), (3000, 250.0, 4), (3000, 250.0, 5000)])
def test_count_alone(n, side, cap, complete):
    print(f"[contacts count] n={n} cap={cap} complete={complete}", flush=True)
    w = gen.uniform_city(n, 8, side, grid_capacity=cap, seed=4)
    g = gen.Generator(w)
    o = Oracle(n, w.box(), w.reach_distance, cap, w.min_meet_time, complete=complete)
    cfg = runtime.make_config(n, w.box(), grid_capacity=cap, record_contacts=True, complete=complete,
                              contact_capacity=1 << 17, unit_capacity=1 << 18)
    with runtime.Workbench(cfg) as wb, runtime.Workbench(cfg) as other:
        for t in range(4):
            xy = g.positions() if t == 0 else g.step()
            o.tick(xy, t)
            want = len(o.contacts())
            wb.set_points(xy, t)
            wb.filter()
            wb.reachability()
            wb.update_meetings()
            assert counts(wb) == (want, want)
            wb.update_schema()
            assert counts(wb) == (want, want)
        other.restore(wb.snapshot())
        n1, n2 = counts(other)
        assert n1 == n2
        trace = runtime.DeviceBuffer(16 * n * 3)
        steps = [g.step() for _ in range(3)]
        trace.upload(np.concatenate([s.reshape(-1) for s in steps]))
        for k, xy in enumerate(steps):
            o.tick(xy, 4 + k)
        want = len(o.contacts())
        for b in (wb, other):
            b.run_ticks(trace.address(0), 4, 3)
            assert counts(b) == (want, want)
        trace.free()
    o.close()
