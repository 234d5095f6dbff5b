"""Every pair of a crowd ends at one tick: more meetings per wave of the table
update than its stage holds, and more per workgroup than one reservation
writes out.  The crowd stands in one spot for ticks 0..6 and is scattered out
of reach at tick 7, so the meetings are all pairs, from 0 to 6, emitted at
tick 7 and at no other; the meeting log ring (also one that wraps) and the
key-value log hold the same."""
import numpy as np
import pytest

from glint_pipeline_amd import runtime

pytestmark = pytest.mark.gpu

N, SIDE = 700, 4000.0
PAIRS = N * (N - 1) // 2


def positions():
    rng = np.random.default_rng(3)
    spot = rng.uniform(0.0, 1.0, (N, 2)) + 2000.0
    g = np.stack(np.meshgrid(np.arange(30), np.arange(30)), axis=-1).reshape(-1, 2)[:N] * 100.0 + 50.0
    return [spot + rng.uniform(-0.1, 0.1, (N, 2)) for _ in range(7)] + [g.astype(np.float64)] * 3


@pytest.mark.parametrize("threads", [256, 512, 1024])
@pytest.mark.parametrize("kv", [False, True])
@pytest.mark.parametrize("ring", [1 << 18, 100_000])
def test_all_pairs_end_at_once(threads, kv, ring):
    print(f"[mass end] threads={threads} kv={kv} ring={ring}", flush=True)
    cfg = runtime.make_config(N, (0.0, 0.0, SIDE, SIDE), grid_capacity=64, min_meet_time=3, table_threads=threads,
                              meeting_log_capacity=ring, kv_capacity=1 << 20 if kv else 0, contact_capacity=1 << 20,
                              num_meeting_buckets=1 << 15)
    want = np.array([(a, b, 0, 6) for a in range(N) for b in range(a + 1, N)], dtype=np.uint32)
    with runtime.Workbench(cfg) as wb:
        for t, xy in enumerate(positions()):
            m = wb.tick(xy, t)
            assert np.array_equal(m, want if t == 7 else want[:0]), f"tick {t}: {len(m)} meetings"
        total, first = wb.meeting_log_info()
        assert (total, first) == (PAIRS, max(0, PAIRS - ring))
        log = wb.meeting_log()
        if first == 0:
            assert np.array_equal(log, want)
        else:   # the newest of them, each once
            assert len(np.unique(log, axis=0)) == ring and (log[:, 2:] == (0, 6)).all()
        if kv:
            assert wb.kv_pending() == 2 * PAIRS
        st = wb.stats()
        assert st["num_active"] == 0 and st["error_flags"] == 0
