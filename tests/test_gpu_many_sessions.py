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
