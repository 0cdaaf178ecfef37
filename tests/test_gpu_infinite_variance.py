"""An update that starts with an infinite variance: nothing is known of one
angle of the LiDAR extrinsic before the scan that estimates it.  P^-1 then
holds zeros in its row and column, and the posterior is the oracle's: x within
the registration tolerances or a hundredth of its deviation (the angle and the
pose are told apart by the pose's prior alone), P within a hundredth."""
import numpy as np
import pytest

from oracle import Oracle, boxminus
from voxelmapplus_fastlio2_amd import Context, LIOConfig, Registrar, initial_covariance, state_vector
from voxelmapplus_fastlio2_amd.synth import QDIAG, ROOM, SEED0, Sequence

pytestmark = pytest.mark.gpu

N = 20000


@pytest.mark.parametrize("max_iter", [1, 5])
@pytest.mark.parametrize("unknown", [6, 7, 8])
def test_unknown_extrinsic_angle_matches_the_oracle(unknown, max_iter):
    cfg = LIOConfig(max_scan_points=N, max_iter=max_iter, estimate_ext=1)
    seq = Sequence(ROOM, SEED0 + 17, N)
    orc, ctx = Oracle(cfg), Context(0)
    s0, P0 = state_vector(*seq.pose(0)), 1e-4 * initial_covariance()
    with Registrar(ctx, cfg) as g:
        orc.set_state(s0, P0)
        orc.build(*seq.scan(0))
        g.set_state(s0, P0)
        g.set_points(*seq.scan(0))
        g.build()
        orc.apply_motion(*seq.motion(1), QDIAG)
        s1, P1 = orc.get_state()
        P1[unknown, unknown] = np.inf
        orc.set_state(s1, P1)
        orc.set_points(*seq.scan(1))
        orc.update()
        so, Po = orc.get_state()
        assert np.isfinite(so).all() and np.isfinite(Po).all()
        g.set_state(s1, P1)
        g.set_points(*seq.scan(1))
        o = g.update()
        sg, Pg = g.get_state()
        assert o.effective > 1000
        assert np.isfinite(sg).all() and np.isfinite(Pg).all()
        d = np.sqrt(np.diag(Po))
        tol = np.full(23, 1e-5)
        tol[[0, 1, 2, 9, 10, 11]] = 1e-4
        assert (np.abs(boxminus(sg, so)) < np.maximum(tol, 0.01 * d)).all()
        assert np.max(np.abs(Pg - Po) / np.outer(d, d)) < 0.01
    ctx.close()
