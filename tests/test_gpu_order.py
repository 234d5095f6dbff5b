"""The order of a tick's meetings as the caller gets them, around the number
from which they are sorted on the device (2048) and at ids that need one bit
more or less: n pairs stand together for ticks 0..2 and part at tick 3, so
tick 3 emits exactly those pairs, in the order of their ids; a second such
tick reuses the buffers, with more or fewer meetings."""
import numpy as np
import pytest

from glint_pipeline_amd import runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npairs", [1, 2047, 2048, 2049, 32_767, 32_768, 32_769, 100_001])
def test_meetings_come_sorted(npairs):
    print(f"[order] {npairs} pairs", flush=True)
    n = 2 * npairs
    k = int(np.ceil(np.sqrt(npairs)))
    side = 14.0 * k + 20.0
    g = np.stack(np.meshgrid(np.arange(k), np.arange(k)), axis=-1).reshape(-1, 2)[:npairs] * 14.0 + 5.0
    perm = np.random.default_rng(npairs).permutation(n)
    a, b = perm[:npairs], perm[npairs:]

    def positions(together):   # the first `together` pairs stand together
        p = np.zeros((n, 2))
        p[a] = g
        p[b] = g + np.where(np.arange(npairs)[:, None] < together, 0.5, 5.0)
        return p

    def want(pairs, start):
        m = np.stack([np.minimum(a, b)[:pairs], np.maximum(a, b)[:pairs]], axis=1)
        m = m[np.lexsort((m[:, 1], m[:, 0]))]
        return np.concatenate([m, np.full((pairs, 1), start), np.full((pairs, 1), start + 2)], axis=1).astype(np.uint32)

    cfg = runtime.make_config(n, (0.0, 0.0, side, side), grid_capacity=200, min_meet_time=1, complete=True)
    with runtime.Workbench(cfg) as wb:
        t = 0
        for pairs in (npairs, max(1, npairs // 2), npairs):
            for step in range(4):
                m = wb.tick(positions(pairs if step < 3 else 0), t)
                w = want(pairs, t - 3) if step == 3 else np.zeros((0, 4), dtype=np.uint32)
                assert np.array_equal(m, w), f"tick {t}: {len(m)} meetings, {len(w)} expected"
                t += 1
