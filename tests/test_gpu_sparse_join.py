"""The join of sparse leaves (one wave per leaf, objects sorted into cells no
smaller than the reach): every tick's contacts, meetings, tested pairs and
active pairs equal the oracle's where it can go wrong:

- one leaf of 2 .. 513 objects: around multiples of the wave, and past the
  most objects a wave takes (the tiles join the leaf then);
- leaf sides around the density below which a leaf is sparse;
- pairs planted just inside and outside the reach, in all directions, across
  cells and on the leaf's edges;
- hundreds of objects in one spot of a wide leaf (more pairs than the stage
  holds at once);
- many leaves with border units, contacts recorded and not (the pruned form),
  in both precisions;
- lon/lat degrees, and a box whose latitudes leave the wave's cells (the
  tiles join its leaves then).
"""
import numpy as np
import pytest

from glint_pipeline_amd import gen, runtime
from tests.parity import run_parity

pytestmark = pytest.mark.gpu

R = 2.0
FP64, GUARD = runtime.PRECISION_FP64, runtime.PRECISION_FP32_GUARD


def planted(n: int, side: float, ticks: int, seed: int, spots: int = 0):
    """Positions of n objects per tick: half anywhere in the box (or in
    `spots` spots), half within 1e-12 to 1e-3 of the reach of one of them,
    inside or outside; a tenth on the box's edges."""
    rng = np.random.default_rng(seed)
    a = (n + 1) // 2
    out = []
    base = rng.uniform(0.0, side, (a, 2))
    if spots:
        base = base[rng.integers(0, min(spots, a), a)] + rng.uniform(-0.3, 0.3, (a, 2))
    for _ in range(ticks):
        base = base + rng.uniform(-0.6, 0.6, (a, 2))
        th = rng.uniform(0.0, 2 * np.pi, n - a)
        th[::3] = np.round(th[::3] / (np.pi / 2)) * (np.pi / 2)
        d = R + rng.choice([-1.0, 1.0], n - a) * 10.0 ** rng.uniform(-12, -3, n - a)
        xy = np.concatenate([base, base[:n - a] + np.stack([d * np.cos(th), d * np.sin(th)], axis=1)])
        edge = rng.random((n, 2)) < 0.05
        xy = np.where(edge, np.round(xy / side) * side, xy)
        out.append(np.clip(xy, 0.0, side).reshape(-1))
    return out


def check(n, side, cap, *, ticks=8, seed=1, spots=0, record=True, precision=FP64, min_meet=1):
    pts = planted(n, side, ticks, seed, spots)
    w = gen.uniform_city(n, ticks, 500.0, grid_capacity=cap, min_meet_time=min_meet)   # (its walk is not used)
    print(f"[sparse] n={n} side={side} cap={cap} precision={precision} record={record}", flush=True)
    return run_parity(w, ticks, check_contacts=record, precision=precision, box=(0.0, 0.0, side, side),
                      positions=lambda t: pts[t], contact_capacity=1 << 20)


@pytest.mark.parametrize("precision", [FP64, GUARD])
@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 127, 128, 129, 511, 512, 513])
def test_one_leaf(n, precision):
    tot = check(n, 400.0, 10 * n, precision=precision, seed=n)
    assert tot["contacts"] > 0 or n < 60


# 200 objects, reach 2: sparse from a side of 2 * sqrt(200 / 0.25) = 56.57 m
@pytest.mark.parametrize("side", [40.0, 56.0, 56.6, 57.0, 8.0e4])
def test_around_the_density(side):
    check(200, side, 2000, record=False, precision=GUARD, seed=7)
    check(200, side, 2000, record=True, precision=FP64, seed=8)


@pytest.mark.parametrize("record", [True, False])
def test_many_objects_in_a_few_spots(record):
    tot = check(400, 500.0, 4000, spots=2, record=record, precision=GUARD, seed=9)
    assert tot["meetings"] > 1000


@pytest.mark.parametrize("precision", [FP64, GUARD])
@pytest.mark.parametrize("record", [True, False])
@pytest.mark.parametrize("cap", [8, 50, 300])
def test_many_leaves(cap, record, precision):
    tot = check(5000, 2500.0, cap, record=record, precision=precision, seed=cap, min_meet=2)
    assert tot["meetings"] > 100


@pytest.mark.parametrize("lat0", [-41.0, 75.0, 88.99])
def test_lonlat(lat0):
    n, side, ticks = 3000, 1500.0, 6
    pts = planted(n, side, ticks, 11)
    proj = runtime.projection_for_box(10.0, lat0)
    fx, fy = proj.deg_per_m_lon, proj.deg_per_m_lat
    deg = [np.stack([10.0 + p.reshape(-1, 2)[:, 0] * fx, lat0 + p.reshape(-1, 2)[:, 1] * fy], axis=1).reshape(-1)
           for p in pts]
    w = gen.uniform_city(n, ticks, side, grid_capacity=40, min_meet_time=1)
    box = (10.0 - fx, lat0 - fy, 10.0 + (side + 1) * fx, lat0 + (side + 1) * fy)
    print(f"[sparse] lon/lat at {lat0}", flush=True)
    tot = run_parity(w, ticks, geography=True, box=box, positions=lambda t: deg[t], contact_capacity=1 << 20)
    assert tot["contacts"] > 100
