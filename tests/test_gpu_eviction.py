"""LRU evictions of one scan against the oracle: the keys in LRU order after
every scan, with few or most of the touched old voxels evicted and created
again in the scan, at the first overflow (room left for some of the
creations), with more touched entries than threads, with a ring whose head
is mostly stale (more of it read than is prefetched), and with more points
than the tables in LDS hold."""
import numpy as np
import pytest

from oracle import Oracle
from voxelmapplus_fastlio2_amd import Context, LIOConfig, Registrar, initial_covariance, state_vector

pytestmark = pytest.mark.gpu

# capacity, points, half extents of the box the points fill (m), move per
# scan (m), scans
CASES = {
    "few_return": (2500, 3000, (10.0, 6.0, 1.0), 3.0, 12),
    "most_return": (16000, 12000, (20.0, 20.0, 2.0), 0.0, 6),
    "one_over": (3700, 2000, (20.0, 20.0, 2.0), 0.0, 4),
    "many_touched": (45000, 30000, (25.0, 25.0, 2.0), 0.0, 4),
    "many_points": (6600, 263000, (7.0, 7.0, 2.0), 2.0, 3),
    "stale_ring": (900, 600, (2.0, 2.0, 2.0), 0.0, 40),
}


def scans(name):
    cap, n, half, move, k = CASES[name]
    rng = np.random.default_rng(len(name) * 1000 + n)
    for q in range(k):
        pts = rng.uniform(-1.0, 1.0, (n - q, 3)) * half
        if name == "stale_ring" and q >= k - 2:  # after a long stand: new ground, more voxels than the map has room for
            pts *= 8.0
        yield state_vector(np.eye(3), [move * q, 0.0, 0.0]), np.ascontiguousarray(pts.T.astype(np.float32))


@pytest.mark.parametrize("name", list(CASES))
def test_evictions_match_the_oracle(name):
    cap, n = CASES[name][:2]
    cfg = LIOConfig(map_capacity=cap, max_scan_points=n)
    orc, ctx = Oracle(cfg), Context(0)
    evicted = 0
    with Registrar(ctx, cfg) as g:
        for k, (s, pts) in enumerate(scans(name)):
            orc.set_state(s, initial_covariance())
            g.set_state(s, initial_covariance())
            g.set_points(*pts)
            if k == 0:
                orc.build(*pts)
                g.build()
            else:
                orc.set_points(*pts)
                orc.map_update()
                evicted += g.map_update().evicted
            a, b = orc.export_map(), g.export_map()
            assert np.array_equal(a["keys"], b["keys"]), f"scan {k}"
            assert np.array_equal(a["ints"][:, 0], b["ints"][:, 0]), f"point counts, scan {k}"
    assert evicted == orc.stats()["evicted"] > 0
    ctx.close()
