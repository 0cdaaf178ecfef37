"""The voxels of a scan in the replay's blocks of 256 against the oracle:
numbers of voxels around a block's edge, walks from one point to past the
longest length class, refits on waves, on lanes and split between the two."""
import numpy as np
import pytest

from mapcmp import compare_maps
from oracle import Oracle
from voxelmapplus_fastlio2_amd import Context, LIOConfig, Registrar, initial_covariance, state_vector

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 9, 23, 24, 61, 62, 63, 64, 130]


def scan(rng, nvox, cfg, shift):
    """nvox voxels of a grid, the i-th with LENGTHS[(i + shift) % 11] points
    scattered near a plane through its centre, in random order."""
    side = int(np.ceil(np.sqrt(nvox)))
    ln = np.array([LENGTHS[(i * 7 + shift) % len(LENGTHS)] for i in range(nvox)])
    v = np.repeat(np.arange(nvox), ln)
    c = np.stack([v % side - side // 2, v // side - side // 2, np.full(len(v), -3)], 1) + 0.5
    p = (c + rng.uniform(-0.45, 0.45, c.shape) * [1.0, 1.0, 0.05]) * cfg.voxel_size
    return np.ascontiguousarray(p[rng.permutation(len(p))].T.astype(np.float32))


@pytest.mark.parametrize("wave_max,long_seg", [(4096, 24), (0, 0), (0, 24)])
@pytest.mark.parametrize("nvox", [1, 255, 256, 257, 800])
def test_blocks_of_voxels_match_the_oracle(nvox, wave_max, long_seg):
    cfg = LIOConfig(max_scan_points=64 * nvox + 256, map_capacity=4 * nvox)
    rng = np.random.default_rng(nvox)
    orc, ctx = Oracle(cfg), Context(0)
    ctx.set_param("replay_wave_max", wave_max)
    ctx.set_param("replay_long_seg", long_seg)
    s = state_vector(np.eye(3), [0.0, 0.0, 0.0])
    with Registrar(ctx, cfg) as g:
        orc.set_state(s, initial_covariance())
        g.set_state(s, initial_covariance())
        for k in range(5):
            pts = scan(rng, nvox, cfg, 3 * k)
            g.set_points(*pts)
            if k == 0:
                orc.build(*pts)
                g.build()
            else:
                orc.set_points(*pts)
                orc.map_update()
                g.map_update()
            r = compare_maps(orc.export_map(), g.export_map())
            margin = r["plane_flag_diff"] + r["merged_flag_diff"]
            assert r["plane_flag_diff"] <= max(2, nvox // 1000), r
            assert max(r["mean_bad"], r["norm_bad"], r["trace_bad"]) <= margin * 8, r
    ctx.close()
