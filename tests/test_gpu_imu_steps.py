"""State and covariance after one package's IMU propagation against the
oracle, for packages of one step to several chunks of 64, at the edges of the
four-step blocks; the covariance is also set to one that is not symmetric.
Both sides sum the same products in double precision, so they agree to a few
hundred roundings of the largest term; 1e-11 of it leaves room for the
factor of the powers of F."""
import numpy as np
import pytest

from oracle import Oracle
from voxelmapplus_fastlio2_amd import Context, ImuConfig, LIOBuilder, LIOConfig
from voxelmapplus_fastlio2_amd.synth import ROOM, SEED0, ImuSequence

pytestmark = pytest.mark.gpu

N = 4000


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 7, 8, 21, 62, 63, 64, 65, 127, 130, 300])
def test_propagation_of_m_samples(m):
    cfg, ic = LIOConfig(max_scan_points=N), ImuConfig()
    seq = ImuSequence(ROOM, SEED0 + 81, N)
    orc, ctx = Oracle(cfg), Context(0)
    orc.imu_config(ic.na, ic.ng, ic.nba, ic.nbg, ic.imu_init_num, ic.gravity_align, np.asarray(ic.r_il).reshape(3, 3),
                   np.asarray(ic.p_il))
    rng = np.random.default_rng(m)
    with LIOBuilder(ctx, cfg) as lb:
        pkg = seq.package(0)
        orc.process(*pkg)
        lb.process(*pkg)
        s, P = lb.reg.get_state()
        s = s.copy()
        P = np.array(P, dtype=np.float64).reshape(23, 23) + 1e-3 * rng.uniform(-1.0, 1.0, (23, 23))
        orc.set_state(s, P)
        lb.reg.set_state(s, P)
        x, y, z, t, _, cs, ce = seq.package(1)
        ts = np.sort(rng.uniform(cs + 1e-4, ce, m))
        acc = np.array([0.0, 0.0, 9.7]) + rng.normal(0.0, 1.0, (m, 3))
        gyro = rng.normal(0.0, 0.4, (m, 3))
        imu = (ts, acc, gyro)
        orc.process(x, y, z, t, imu, cs, ce)
        lb.process(x, y, z, t, imu, cs, ce)
        so, Po = orc.get_state()
        sg, Pg = lb.reg.get_state()
        assert np.abs(so - sg).max() <= 1e-11 * np.abs(so).max()
        assert np.abs(np.asarray(Po) - np.asarray(Pg)).max() <= 1e-11 * np.abs(Po).max()
    ctx.close()
