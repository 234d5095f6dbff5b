"""The grouping of a tick's contacts around the size that one workgroup takes
whole (12288 list entries) and the number of regions it can tell apart
(2048): a crowd of k objects has k(k-1)/2 pairs, 12246 of 157 objects, 12403
of 158, beside objects far apart.  Meetings, active pairs and contacts of
every tick equal the oracle's."""
import numpy as np
import pytest

from tests.parity import run_positions_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("buckets", [1, 1 << 12, 1 << 22, 1 << 23])
@pytest.mark.parametrize("crowd", [0, 2, 50, 156, 157, 158, 159, 230])
def test_lists_around_one_tile(crowd, buckets):
    print(f"[bucketing] crowd {crowd} buckets {buckets}", flush=True)
    rng = np.random.default_rng(crowd)
    apart = np.stack(np.meshgrid(np.arange(20), np.arange(20)), axis=-1).reshape(-1, 2) * 40.0 + 20.0
    xys = []
    for t in range(7):
        p = apart + rng.uniform(-1.0, 1.0, apart.shape)
        if t != 5:   # the crowd parts for a tick
            p[:crowd] = 400.0 + rng.uniform(0.0, 1.0, (crowd, 2))
        xys.append(p.reshape(-1))
    for record in (False, True):
        run_positions_parity(xys, (0.0, 0.0, 800.0, 800.0), grid_capacity=300, min_meet=2, num_meeting_buckets=buckets,
                             contact_capacity=1 << 16, record_contacts=record)


@pytest.mark.parametrize("bits", [7, 8, 9, 11, 12, 19, 20, 21])
def test_numbers_of_regions(bits):
    """2^bits regions: 256 coarse bins, fewer with fewer regions, more past
    2^19 of them; 26335 pairs, more than one workgroup takes whole."""
    print(f"[bucketing] 2^{bits} regions", flush=True)
    rng = np.random.default_rng(bits)
    xys = [(400.0 + rng.uniform(0.0, 1.0, (230, 2)) + (np.arange(230)[:, None] % 7 == t) * 30.0).reshape(-1)
           for t in range(7)]
    for record in (False, True):
        run_positions_parity(xys, (0.0, 0.0, 800.0, 800.0), grid_capacity=300, min_meet=2,
                             num_meeting_buckets=1 << (bits + 11), contact_capacity=1 << 16, record_contacts=record)
