"""Leaves of more reaches across than single-precision offsets in reaches can
hold (3.4e38): pairs at one point, or within reach of each other, are contacts
there as in any other leaf, and every tick equals the oracle's."""
import numpy as np
import pytest

from glint_pipeline_amd import gen
from tests.parity import run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reach,side", [(2.0, 400.0), (1e-12, 400.0), (1e-30, 400.0), (1e-40, 400.0), (1e-300, 400.0),
                                        (2.0, 1e20), (2.0, 1e39), (2.0, 1e45)])
@pytest.mark.parametrize("record", [True, False])
def test_reaches_across_a_leaf(reach, side, record):
    n, ticks = 200, 6
    rng = np.random.default_rng(3)
    # half the objects over the box and half near its low corner, where
    # coordinates are fine enough for any reach; every point held by up to two
    spots = np.concatenate([rng.uniform(0.0, side, (50, 2)), rng.uniform(0.0, 8.0 * reach, (50, 2))])
    pts = [np.repeat(spots[rng.permutation(100)] if t == 3 else spots, 2, axis=0).reshape(-1) for t in range(ticks)]
    w = gen.uniform_city(n, ticks, 500.0, grid_capacity=2 * n, min_meet_time=1, reach_distance=reach)   # (its walk is not used)
    print(f"[sparse extent] reach {reach} side {side} record {record}", flush=True)
    tot = run_parity(w, ticks, check_contacts=record, box=(0.0, 0.0, side, side), positions=lambda t: pts[t],
                     contact_capacity=1 << 16)
    assert tot["contacts"] >= 100 * ticks or not record
