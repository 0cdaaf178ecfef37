"""Acting merge candidates of a batch whose sessions begin and end around the
2,048-point tiles of their compaction, empty scans among them: posterior and
map bitwise as each session alone."""
import numpy as np
import pytest

from voxelmapplus_fastlio2_amd import Context, LIOConfig, Registrar, initial_covariance, register_batch, state_vector
from voxelmapplus_fastlio2_amd.synth import ROOM, SEED0, Sequence

pytestmark = pytest.mark.gpu

N = 12000


def start(ctx, seq):
    g = Registrar(ctx, LIOConfig(max_scan_points=N, map_capacity=40000))
    R, t = seq.pose(0)
    g.set_state(state_vector(R, t), initial_covariance())
    g.set_points(*seq.scan(0))
    g.build()
    return g


@pytest.mark.parametrize("sizes", [(2048,), (2049,), (0, 2047, 1, 0), (2048, 0, 0, 2048), (N, 0, 5000, 2047, 0, 3)])
def test_acting_candidates_of_a_batch(sizes):
    a, b = Context(0), Context(0)
    seqs = [Sequence(ROOM, SEED0 + 300 + i, N) for i in range(len(sizes))]
    alone, batch = [start(a, q) for q in seqs], [start(b, q) for q in seqs]
    merges = 0
    for k in range(1, 12):
        for i, n in enumerate(sizes):
            m = n if k % 4 == 0 else N  # whole scans in between, so that planes freeze and merge
            for g in (alone[i], batch[i]):
                R, t = seqs[i].pose(k)
                g.set_state(state_vector(R, t), initial_covariance())
                g.set_points(*(v[:m].copy() for v in seqs[i].scan(k)))
        for g in alone:
            merges += g.register()[1].merges
        register_batch(batch)
        for i, (x, y) in enumerate(zip(alone, batch)):
            for u, v in zip(x.get_state(), y.get_state()):
                assert np.array_equal(u, v), (k, i)
            ex, ey = x.export_map(), y.export_map()
            assert all(np.array_equal(ex[f], ey[f]) for f in ex), (k, i)
    assert merges > 0
    for g in alone + batch:
        g.close()
    a.close()
    b.close()
