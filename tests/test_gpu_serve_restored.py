"""A snapshot restored under a server: its queries read the log that came with
the snapshot, also where the restored tick is the server's own (the bounds of
the log kept from the server's tick are not those of the restored one)."""
import numpy as np
import pytest

from glint_pipeline_amd import runtime

pytestmark = pytest.mark.gpu

N, SIDE, LAST = 400, 4000.0, 9
CFG = dict(grid_capacity=64, min_meet_time=3, meeting_log_capacity=1 << 16, contact_capacity=1 << 18)


def positions(tick, crowd):
    g = np.stack(np.meshgrid(np.arange(20), np.arange(20)), axis=-1).reshape(-1, 2)[:N] * 100.0 + 50.0
    xy = g.astype(np.float64)
    if tick <= 6:   # they stand together for ticks 0..6
        xy[:crowd] = 2000.0 + np.random.default_rng(tick).uniform(0.0, 0.9, (crowd, 2))
    return xy


@pytest.mark.parametrize("hops", [1, 2])
@pytest.mark.parametrize("block_ticks", [4, 0xFFFFFFFF])
@pytest.mark.parametrize("other", [0, 30])
def test_queries_after_a_restore(other, block_ticks, hops):
    print(f"[serve restored] {other} together, index blocks of {block_ticks} ticks, {hops} hops", flush=True)
    with runtime.Workbench(runtime.make_config(N, (0.0, 0.0, SIDE, SIDE), **CFG)) as wb:
        for t in range(LAST + 1):
            wb.tick(positions(t, other), t)
        snap = wb.snapshot()
    # (the server and then its context are closed whatever fails)
    with runtime.Workbench(runtime.make_config(N, (0.0, 0.0, SIDE, SIDE), **CFG)) as wb, \
            runtime.Server(wb, arena_bytes=1 << 28, index_block_ticks=block_ticks) as sv:
        bufs = []
        for t in range(LAST + 1):
            bufs.append(runtime.DeviceBuffer(16 * N))
            bufs[-1].upload(positions(t, 60))
            sv.tick(t, d_full_xy=bufs[-1].address())
        q = sv.submit([1, 2], 0, LAST, hops)
        sv.drain()
        h1, _ = sv.result(q)
        assert len(h1) == 2 * 59
        wb.restore(snap)
        total, first = wb.meeting_log_info()
        assert (total, first) == (other * (other - 1) // 2, 0)
        # the server sealed its own 1770 meetings in blocks, where it has any:
        # without blocks the log alone answers
        q = sv.submit([1, 2], 0, LAST, hops)
        sv.drain()
        h1, _ = sv.result(q)
        if block_ticks == 0xFFFFFFFF:
            assert len(h1) == (2 * (other - 1) if other else 0)
    for b in bufs:
        b.free()
