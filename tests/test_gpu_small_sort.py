"""Maps of scans around the edges of a sort tile (2,048 points) and of its waves
against the oracle: keys in LRU order and point counts after every scan."""
import numpy as np
import pytest

from oracle import Oracle
from voxelmapplus_fastlio2_amd import Context, LIOConfig, Registrar, initial_covariance, state_vector

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 511, 513, 2047, 2048, 2049, 4097])
def test_scans_around_a_tile(n):
    cfg = LIOConfig(max_scan_points=n, map_capacity=3 * n)
    rng = np.random.default_rng(n)
    orc, ctx = Oracle(cfg), Context(0)
    s = state_vector(np.eye(3), [0.0, 0.0, 0.0])
    with Registrar(ctx, cfg) as g:
        orc.set_state(s, initial_covariance())
        g.set_state(s, initial_covariance())
        for k in range(4):
            p = rng.normal(0.0, 1.0 + k, (3, n)).astype(np.float32)
            p[:, n // 2 :] = p[:, : n - n // 2]  # repeated voxels, in another order
            g.set_points(*p)
            if k == 0:
                orc.build(*p)
                g.build()
            else:
                orc.set_points(*p)
                orc.map_update()
                g.map_update()
            a, b = orc.export_map(), g.export_map()
            assert np.array_equal(a["keys"], b["keys"]), k
            assert np.array_equal(a["ints"][:, 0], b["ints"][:, 0]), k
    ctx.close()
