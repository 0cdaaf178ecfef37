"""Device point sets are refused for a value that is not finite, or a time
before its predecessor's, at any place, around the edges of the check's blocks
(1,024 points) and of its threads; equal times and the last finite values are
accepted."""
import numpy as np
import pytest
import torch

from voxelmapplus_fastlio2_amd import Context, LIOBuilder, LIOConfig, VmpError
from voxelmapplus_fastlio2_amd.synth import ROOM, SEED0, ImuSequence

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1023, 1024, 1025, 5000])
def test_check_of_device_points(n):
    seq, ctx = ImuSequence(ROOM, SEED0 + 90, 5000), Context(0)
    with LIOBuilder(ctx, LIOConfig(max_scan_points=5000)) as lb:
        lb.process(*seq.package(0))
        lb.process(*seq.package(1))
        x, y, z, t, imu, cs, ce = seq.package(2)
        good = np.stack([x, y, z, np.minimum.accumulate(t[::-1])[::-1]])[:, :n].astype(np.float32)
        good[3, n // 2 :] = good[3, -1]  # equal times

        def run(a):
            dev = torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
            torch.cuda.synchronize()
            lb.reg.set_raw_device(*(dev[k].data_ptr() for k in range(4)), n, imu, cs, ce)
            return lb.reg.register()

        before = [v.copy() for v in lb.reg.get_state()]
        for i in sorted({0, 1, n // 2, n - 2, n - 1} & set(range(n))):
            for row, bad in ((0, np.nan), (1, np.inf), (2, -np.inf), (3, np.nan), (3, None)):
                a = good.copy()
                if bad is None:
                    if i == 0:
                        continue
                    a[3, i] = np.nextafter(a[3, i - 1], np.float32(-1.0))
                else:
                    a[row, i] = bad
                with pytest.raises(VmpError, match="-1"):
                    run(a)
        for u, v in zip(before, lb.reg.get_state()):
            assert np.array_equal(u, v)
        run(good)
    ctx.close()
