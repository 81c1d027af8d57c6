"""The tracking loop's 512-thread form (FP64 sums) at the image sizes where its
split changes: fewer pixels than one workgroup, one row more or less than whole
workgroups, chunks that are not a multiple of the workgroup, and the bound on
the number of workgroups; with one and with four pixels per thread.

One Gauss-Newton iteration in all, at one level, so that both sides sum the
same pixels: the number of pixels summed is the oracle's, and the poses differ
by the order of an FP64 sum alone (1e-16 x the sums' condition, far below the
1e-6 allowed, which covers the float rounding of the solved system).
"""
import numpy as np
import pytest

from helpers import B, sys_cfg, synth, to_dev
from oracle import binding as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,rows", [
    (96, 64),      # level 2: 24 x 16 = 384 pixels, fewer than a workgroup
    (129, 97),     # odd sizes at every level
    (321, 255),    # 81855 pixels: 160 chunks of 512, the last one short
    (723, 541),    # 391143 pixels: 256 chunks of 1528
    (1024, 512)])  # 256 chunks of exactly 4 pixels per thread
@pytest.mark.parametrize("level", [0, 1, 2])
@pytest.mark.parametrize("spread", [1, 0])
def test_one_iteration_sums_the_oracles_pixels(dev, cols, rows, level, spread):
    f = 0.82 * cols
    c = dict(cols=cols, rows=rows, f=f, cx=0.5 * (cols - 1), cy=0.5 * (rows - 1), voxel=0.01,
             trunc=0.03, buckets=1 << 18, blocks=100000)
    cfg = sys_cfg(c)
    cfg.icp_spread = spread
    cfg.icp_thresh = 1.0  # the oracle's own residual at 24 x 16 is above the default's 1e-4
    for i in range(3):
        cfg.icp_iters[i] = 1 if i == level else 0
        cfg.icp_min_count[i] = 1
    g, o, s = B.System(cfg), O.OracleSystem(cfg), synth(c)
    for i in range(2):
        d, rgb, lab = s.render(i)
        g.grab(to_dev(d, dev), to_dev(rgb, dev), to_dev(lab, dev))
        rg, ro = g.result(), o.grab(d, rgb, lab)
        assert rg["tracked"] == ro["tracked"], (rg, ro)
        assert rg["icp_count"] == ro["icp_count"], (rg, ro)
        assert np.abs(rg["pose"] - ro["pose"]).max() < 1e-6
    assert ro["icp_count"] > 0  # at 24 x 16 the frame itself is lost, on both sides
