"""Batches of many small sessions: a few of them with merge candidates and
long runs of sessions without any before, between and behind them."""
import numpy as np
import pytest

from voxelmapplus_fastlio2_amd import Context, LIOConfig, Registrar, initial_covariance, register_batch, state_vector
from voxelmapplus_fastlio2_amd.synth import ROOM, SEED0, Sequence

pytestmark = pytest.mark.gpu

N, SMALL = 12000, 40


def start(ctx, seq, n):
    g = Registrar(ctx, LIOConfig(max_scan_points=n, map_capacity=30000 if n == N else 2000))
    g.set_state(state_vector(*seq.pose(0)), initial_covariance())
    g.set_points(*(v[:n].copy() for v in seq.scan(0)))
    g.build()
    return g


# sessions with whole scans; the runs between them are around the 16 sessions
# that one thread takes, longer than a block's 256 threads, and empty
@pytest.mark.parametrize("count,large", [(150, [0, 16, 32, 49, 50, 149]), (330, [15, 310]), (40, []), (300, [299])])
def test_sessions_without_candidates_between_those_with(count, large):
    a, b = Context(0), Context(0)
    size = [N if i in large else SMALL for i in range(count)]
    seqs = {i: Sequence(ROOM, SEED0 + 500 + i, N) for i in set(large) | {-1}}
    seq = [seqs.get(i, seqs[-1]) for i in range(count)]
    batch = [start(b, seq[i], size[i]) for i in range(count)]
    watched = sorted(set(large) | {0, count // 2, count - 1})
    alone = {i: start(a, seq[i], size[i]) for i in watched}
    merges = 0
    for k in range(1, 10):
        for i, g in list(enumerate(batch)) + list(alone.items()):
            g.set_state(state_vector(*seq[i].pose(k)), initial_covariance())
            g.set_points(*(v[: size[i]].copy() for v in seq[i].scan(k)))
        register_batch(batch)
        for i, g in alone.items():
            merges += g.register()[1].merges
            for u, v in zip(g.get_state(), batch[i].get_state()):
                assert np.array_equal(u, v), (k, i)
            ex, ey = g.export_map(), batch[i].export_map()
            assert all(np.array_equal(ex[f], ey[f]) for f in ex), (k, i)
    assert merges > 0 or not large
    for g in batch + list(alone.values()):
        g.close()
    a.close()
    b.close()


def test_states_of_a_large_batch():
    """The covariances of a batch of more than 64 sessions are fetched when one
    is asked for: every state bitwise as from batches of at most 64, before and
    after a change, another step, a larger workspace and a step without them."""
    n, count = 300, 70
    a, b = Context(0), Context(0)
    seq = [Sequence(ROOM, SEED0 + 700 + i % 5, n) for i in range(count)]
    small, large = [start(a, q, n) for q in seq], [start(b, q, n) for q in seq]
    qdiag = np.full(23, 1e-5)

    def check(which):
        for i in which:
            for u, v in zip(small[i].get_state(), large[i].get_state()):
                assert np.array_equal(u, v), i

    def scans(k, which):
        for i in which:
            for g in (small[i], large[i]):
                g.apply_motion(*seq[i].motion(k), qdiag)
                g.set_points(*(v[:n].copy() for v in seq[i].scan(k)))

    def step(k, which):
        scans(k, which)
        register_batch([large[i] for i in which])
        for lo in range(0, len(which), 64):
            register_batch([small[i] for i in which[lo : lo + 64]])

    everyone = list(range(count))
    check(everyone)
    step(1, everyone)
    check([69, 0, 33])
    check(everyone)
    for g in (small[5], large[5]):  # a change of one session
        g.apply_motion(*seq[5].motion(2), qdiag)
    for g in (small[6], large[6]):
        g.set_state(state_vector(*seq[6].pose(2)))
    check(everyone)
    step(3, everyone[:66])  # large again, without some
    check(everyone)
    step(4, everyone)
    step(5, everyone[10:20])  # a small one behind it
    check(everyone)
    step(6, everyone)
    b.reserve(n * 100, 100)
    check(everyone)
    step(7, everyone)
    scans(8, everyone)  # priors of all behind the step
    check(everyone)
    for g in small + large:
        g.close()
    a.close()
    b.close()
