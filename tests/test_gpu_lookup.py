"""The lookup's walk, shared by the objects of a wave: every tick's contacts,
meetings, tested pairs and drop counts equal the oracle's where it can go
wrong.  The box is a hundred times as high as wide, so a leaf twice the reach
high is a twentieth of it wide and an object selects up to hundreds of leaves:
the second pass over an object's leaves, and more branches to visit than the
wave's stack takes at full width.  Numbers of objects around the wave."""
import numpy as np
import pytest

from glint_pipeline_amd import gen, runtime
from tests.parity import run_parity

pytestmark = pytest.mark.gpu


def crowd(n: int, ticks: int, seed: int):
    rng = np.random.default_rng(seed)
    xy = rng.uniform(0.0, 1.0, (n, 2)) * (4.0, 20.0) + (28.3, 2990.3)
    out = []
    for _ in range(ticks):
        out.append(np.clip(xy, (0.0, 0.0), (60.0, 6000.0)).reshape(-1))
        xy = xy + rng.uniform(-0.2, 0.2, (n, 2))
    return out


@pytest.mark.parametrize("complete", [False, True])
@pytest.mark.parametrize("n,cap", [(63, 1), (65, 1), (700, 1), (1500, 2), (1500, 8)])
def test_narrow_leaves(n, cap, complete):
    ticks = 4
    pts = crowd(n, ticks, n)
    w = gen.uniform_city(n, ticks, 500.0, grid_capacity=cap, min_meet_time=1)   # (its walk is not used)
    print(f"[lookup] n={n} cap={cap} complete={complete}", flush=True)
    tot = run_parity(w, ticks, complete=complete, box=(0.0, 0.0, 60.0, 6000.0), positions=lambda t: pts[t],
                     unit_capacity=1 << 20, node_capacity=1 << 15, contact_capacity=1 << 21)
    assert tot["contacts"] > n


def test_narrow_leaves_lonlat():
    n, ticks = 700, 4
    pts = crowd(n, ticks, 5)
    proj = runtime.projection_for_box(10.0, 40.0)
    fx, fy = proj.deg_per_m_lon, proj.deg_per_m_lat
    deg = [np.stack([10.0 + p.reshape(-1, 2)[:, 0] * fx, 40.0 + p.reshape(-1, 2)[:, 1] * fy], axis=1).reshape(-1)
           for p in pts]
    w = gen.uniform_city(n, ticks, 500.0, grid_capacity=2, min_meet_time=1)
    print("[lookup] lon/lat", flush=True)
    tot = run_parity(w, ticks, geography=True, box=(10.0, 40.0, 10.0 + 60.0 * fx, 40.0 + 6000.0 * fy),
                     positions=lambda t: deg[t], unit_capacity=1 << 20, node_capacity=1 << 15,
                     contact_capacity=1 << 21)
    assert tot["contacts"] > n
