"""vmp_state_get after calls that change the state while a submitted batch is
in flight: the state behind the change, bitwise the one of a session that
registers and changes without overlap, however the batch is completed."""
import numpy as np
import pytest

from voxelmapplus_fastlio2_amd import (
    Context,
    LIOConfig,
    Registrar,
    apply_motion_batch,
    initial_covariance,
    register_batch_submit,
    register_batch_wait,
    state_vector,
)
from voxelmapplus_fastlio2_amd.synth import QDIAG, ROOM, SEED0, Sequence

pytestmark = pytest.mark.gpu

N = 3000


def start(ctx, seq):
    g = Registrar(ctx, LIOConfig(max_scan_points=N, map_capacity=20000))
    g.set_state(state_vector(*seq.pose(0)), initial_covariance())
    g.set_points(*seq.scan(0))
    g.build()
    return g


@pytest.mark.parametrize("complete", ["wait", "next_step"])
@pytest.mark.parametrize("change", ["apply_motion", "apply_motion_batch", "set_state", "set_x_only", "none"])
def test_state_behind_a_change_in_flight(change, complete):
    seq = Sequence(ROOM, SEED0 + 901, N)
    dR, dp = seq.motion(2)

    def apply(g):
        if change == "apply_motion":
            g.apply_motion(dR, dp, QDIAG)
        elif change == "apply_motion_batch":
            apply_motion_batch([g], [dR], [dp], QDIAG)
        elif change == "set_state":
            g.set_state(state_vector(*seq.pose(2)), 2.0 * initial_covariance())
        elif change == "set_x_only":
            g.set_state(state_vector(*seq.pose(2)))

    ctx_a, ctx_b = Context(0), Context(0)
    alone, over, other = start(ctx_a, seq), start(ctx_b, seq), start(ctx_b, seq)
    for g in (alone, over, other):
        g.apply_motion(*seq.motion(1), QDIAG)
        g.set_points(*seq.scan(1))
    alone.register()
    want_0 = alone.get_state()
    apply(alone)
    want = alone.get_state()
    assert change == "none" or not np.array_equal(want_0[0], want[0])

    register_batch_submit([over])
    apply(over)
    if complete == "wait":
        register_batch_wait(ctx_b, 1)
    else:
        other.register()  # completes the submitted batch first
    for _ in range(2):
        got = over.get_state()
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    for u, v in zip(over.odom(), alone.odom()):
        assert np.array_equal(u, v)

    # the next step starts from it, and hands its own result out again
    for g in (alone, over):
        g.set_points(*seq.scan(2))
        g.register()
    for u, v in zip(over.get_state(), alone.get_state()):
        assert np.array_equal(u, v)
    for g in (alone, over, other):
        g.close()
    ctx_a.close()
    ctx_b.close()
