"""vmp_state_apply_motion_batch while a submitted batch runs returns without
waiting for that batch, also where nothing between two priors waits for the
stream (device buffers whose check is switched off)."""
import time

import numpy as np
import pytest
import torch

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
from voxelmapplus_fastlio2_amd.synth import QDIAG, SEED0, STREET, Sequence

pytestmark = pytest.mark.gpu

N, S, SCANS = 60000, 12, 8


@pytest.mark.parametrize("check", [0, 1])
def test_prior_of_the_next_batch_does_not_wait(check):
    ctx = Context(0)
    ctx.set_param("check_points", check)
    seqs = [Sequence(STREET, SEED0 + 950 + i, N) for i in range(S)]
    regs = [Registrar(ctx, LIOConfig(max_scan_points=N, map_capacity=150000)) for _ in seqs]
    dev = [[torch.from_numpy(np.stack(q.scan(k))).to("cuda:0") for k in range(SCANS)] for q in seqs]
    torch.cuda.synchronize()
    ctx.reserve(N * S, S)
    motion = [None] + [[q.motion(k) for q in seqs] for k in range(1, SCANS)]
    for q, g, d in zip(seqs, regs, dev):
        g.set_state(state_vector(*q.pose(0)), initial_covariance())
        g.set_points_device(d[0][0].data_ptr(), d[0][1].data_ptr(), d[0][2].data_ptr(), N)
        g.build()

    def prior(k):
        apply_motion_batch(regs, [a for a, _ in motion[k]], [b for _, b in motion[k]], QDIAG)

    prior(1)
    shares = []
    for k in range(1, SCANS):
        for g, d in zip(regs, dev):
            g.set_points_device(d[k][0].data_ptr(), d[k][1].data_ptr(), d[k][2].data_ptr(), N)
        register_batch_submit(regs)  # completes batch k - 1
        t0 = time.perf_counter()
        if k + 1 < SCANS:
            prior(k + 1)
        t1 = time.perf_counter()
        register_batch_wait(ctx, S)
        t2 = time.perf_counter()
        if 1 < k < SCANS - 1:
            shares.append((t1 - t0) / (t2 - t0))
    print("prior's share of the time to the batch's end:", [f"{s:.2f}" for s in shares], flush=True)
    # it has waited for the batch where it takes nearly all of that time
    assert np.median(shares) < 0.6, shares
    for g in regs:
        g.close()
    ctx.close()
