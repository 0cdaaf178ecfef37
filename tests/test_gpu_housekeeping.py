"""Hash table rebuilds and LRU ring compactions against the oracle: the voxel
keys in LRU order after every scan, for maps that stay full while the sensor
moves on (tombstones pile up), over one-layer maps (four of a line's eight
slots), and for more sessions in one step than one rebuild launch lists."""
import numpy as np
import pytest

from oracle import Oracle
from voxelmapplus_fastlio2_amd import Context, LIOConfig, Registrar, initial_covariance, register_batch, state_vector

pytestmark = pytest.mark.gpu


def floor_scan(rng, n, layers):
    """n points on `layers` voxel layers, 12 m x 8 m around the sensor."""
    p = rng.uniform([-6.0, -4.0, 0.0], [6.0, 4.0, 1.0], (n, 3))
    p[:, 2] = -1.3 + 0.5 * np.floor(p[:, 2] * layers) + 0.02 * rng.standard_normal(n)
    return np.ascontiguousarray(p.T.astype(np.float32))


def pose(k, s=0):
    return state_vector(np.eye(3), [0.7 * k, 3.0 * s, 0.0])


@pytest.mark.parametrize("capacity,n,layers,step", [(600, 500, 1, 4.0), (1000, 900, 8, 1.0), (380, 130, 1, 0.5)])
def test_full_map_rebuilds_match_the_oracle(capacity, n, layers, step):
    cfg = LIOConfig(map_capacity=capacity, max_scan_points=n)
    rng = np.random.default_rng(capacity + n + layers)
    orc, ctx = Oracle(cfg), Context(0)
    rebuilt = 0
    with Registrar(ctx, cfg) as g:
        for k in range(40):
            pts = floor_scan(rng, n if k % 3 else n - 7, layers)
            s = pose(step * k)
            orc.set_state(s, initial_covariance())
            g.set_state(s, initial_covariance())
            g.set_points(*pts)
            if k == 0:
                orc.build(*pts)
                g.build()
                continue
            orc.set_points(*pts)
            orc.map_update()
            rebuilt += g.map_update().maintenance & 1
            assert np.array_equal(orc.export_map()["keys"], g.export_map()["keys"]), f"scan {k}"
    assert rebuilt >= 1 and orc.stats()["evicted"] > capacity
    ctx.close()


def test_rebuilds_of_many_sessions_in_one_step():
    """64 sessions whose tables fill up in the same steps (one rebuild launch
    lists 60); three of them against the same sessions alone."""
    cfg = LIOConfig(map_capacity=150, max_scan_points=120)
    ctx = Context(0)
    regs = [Registrar(ctx, cfg) for _ in range(67)]
    alone = {0: 64, 59: 65, 63: 66}
    rngs = [np.random.default_rng(900 + i) for i in range(64)]
    most = 0
    for k in range(16):
        scans = [floor_scan(r, 120, 4) for r in rngs]
        for i in list(range(64)) + list(alone):
            for reg in [regs[i]] + ([regs[alone[i]]] if i in alone else []):
                reg.set_state(pose(k, i), 1e-6 * initial_covariance())
                reg.set_points(*scans[i])
        if k == 0:
            for reg in regs:
                reg.build()
            continue
        _, m = register_batch(regs[:64])
        most = max(most, sum(q.maintenance & 1 for q in m))
        for i, a in alone.items():
            regs[a].register()
            x, y = regs[i].export_map(), regs[a].export_map()
            assert all(np.array_equal(x[f], y[f]) for f in x), (k, i)
    assert most > 60
    for reg in regs:
        reg.close()
    ctx.close()
