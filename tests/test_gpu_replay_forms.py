"""The forms of the replay (a refitting voxel per wave, per lane, the long ones
per wave and the rest per lane) give the same map, bit for bit, and the oracle's
decisions: every plane and every merge.  The points are the oracle's own (the
pose is the identity), so a decision can differ only where the roundings of an
eigenvalue or of a gate, 1e-7 of their size at most, straddle a threshold: the
voxels here lie 200 times below the plane threshold, and none of the few
thousand gates of these seeds is expected that close to its bound."""
import numpy as np
import pytest

from mapcmp import compare_maps
from oracle import Oracle
from test_gpu_replay_order import scan
from voxelmapplus_fastlio2_amd import Context, LIOConfig, Registrar, initial_covariance, state_vector

pytestmark = pytest.mark.gpu

FORMS = [(4096, 24), (0, 0), (0, 24), (0, 62)]  # replay_wave_max, replay_long_seg


@pytest.mark.parametrize("nvox", [1, 255, 256, 257, 800])
def test_forms_agree_and_decide_as_the_oracle(nvox):
    cfg = LIOConfig(max_scan_points=64 * nvox + 256, map_capacity=4 * nvox)
    s = state_vector(np.eye(3), [0.0, 0.0, 0.0])
    orc = Oracle(cfg)
    orc.set_state(s, initial_covariance())
    ctxs, regs = [], []
    for wave_max, long_seg in FORMS:
        ctx = Context(0)
        ctx.set_param("replay_wave_max", wave_max)
        ctx.set_param("replay_long_seg", long_seg)
        ctxs.append(ctx)
        regs.append(Registrar(ctx, cfg))
        regs[-1].set_state(s, initial_covariance())
    rng = np.random.default_rng(1000 + nvox)
    for k in range(5):
        pts = scan(rng, nvox, cfg, 3 * k)
        if k == 0:
            orc.build(*pts)
        else:
            orc.set_points(*pts)
            orc.map_update()
        maps = []
        for g in regs:
            g.set_points(*pts)
            if k == 0:
                g.build()
            else:
                g.map_update()
            maps.append(g.export_map())
        for form, m in zip(FORMS[1:], maps[1:]):
            for key in m:
                assert np.array_equal(m[key], maps[0][key]), (form, k, key)
        r = compare_maps(orc.export_map(), maps[0])
        assert r["plane_flag_diff"] == 0 and r["merged_flag_diff"] == 0, (k, r)
        assert max(r["mean_bad"], r["norm_bad"], r["trace_bad"]) == 0, (k, r)
    assert r["merged"] > nvox // 2 or nvox == 1
    for g in regs:
        g.close()
    for ctx in ctxs:
        ctx.close()
