"""The meeting log ring where a tick's meetings wrap it never, once and
thousands of times: a crowd's pairs end together at two ticks, and the log
holds the newest of them, each once."""
import numpy as np
import pytest

from glint_pipeline_amd import runtime

pytestmark = pytest.mark.gpu

N = 300
PAIRS = N * (N - 1) // 2


@pytest.mark.parametrize("kv", [False, True])
@pytest.mark.parametrize("threads", [256, 512, 1024])
@pytest.mark.parametrize("ring", [1, 3, 1000, PAIRS - 1, PAIRS, PAIRS + 1, 2 * PAIRS - 1, 2 * PAIRS])
def test_newest_meetings(ring, threads, kv):
    print(f"[log ring] {ring} of 2 x {PAIRS}, {threads} threads, kv {kv}", flush=True)
    rng = np.random.default_rng(3)
    apart = np.stack(np.meshgrid(np.arange(20), np.arange(20)), axis=-1).reshape(-1, 2)[:N] * 100.0 + 50.0
    cfg = runtime.make_config(N, (0.0, 0.0, 2000.0, 2000.0), grid_capacity=64, min_meet_time=3, table_threads=threads,
                              meeting_log_capacity=ring, kv_capacity=1 << 19 if kv else 0, contact_capacity=1 << 19)
    pairs = np.array([(a, b) for a in range(N) for b in range(a + 1, N)], dtype=np.uint32)
    with runtime.Workbench(cfg) as wb:
        for t in range(14):
            together = t % 7 < 5
            xy = rng.uniform(0.0, 0.9, (N, 2)) + 777.0 if together else apart
            m = wb.tick(np.ascontiguousarray(xy).reshape(-1), t)
            assert len(m) == (PAIRS if t in (5, 12) else 0)
        total, first = wb.meeting_log_info()
        assert (total, first) == (2 * PAIRS, 2 * PAIRS - ring)
        log = wb.meeting_log()
    assert len(log) == ring and len(np.unique(log, axis=0)) == ring
    newest = log[log[:, 2] == 7]
    assert len(newest) == min(ring, PAIRS) and (newest[:, 3] == 11).all()
    assert (log[log[:, 2] != 7][:, 2:] == (0, 4)).all()
    if ring >= PAIRS:
        assert np.array_equal(newest[:, :2], pairs)
