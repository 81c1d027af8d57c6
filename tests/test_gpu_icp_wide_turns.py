"""The tracking loop's 512-thread form (FP64 sums) where test_gpu_icp_wide.py
does not reach: chunks so long that a workgroup takes its pixels in several turns
(the last one short), chunks of which the three-slot copy of the pass uses two
slots, and the photometric term at all of them, whose records and row pass follow
the same split.

As there: one Gauss-Newton iteration in all, at one level; the numbers of pixels
summed, of both terms, are the oracle's, and the poses differ by the order of the
FP64 sums alone, far below the 1e-6 allowed for the float rounding of the solved
system.
"""
import numpy as np
import pytest

from helpers import B, sys_cfg, synth, to_dev
from oracle import binding as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,rows,level", [
    (1279, 719, 0),  # 919601 pixels: 256 chunks of 3593, two turns of four slots
    (1279, 719, 1),  # 639 x 359: 256 chunks of 897
    (480, 360, 0),   # 256 chunks of 675, or (spread 0) 85 of 2033
    (321, 255, 0),   # 160 chunks of 512, the last one short
    (321, 255, 1),   # 160 x 127: 40 chunks of 508
    (723, 541, 0)])  # 256 chunks of 1528
@pytest.mark.parametrize("icp_only", [1, 0])
@pytest.mark.parametrize("spread", [1, 0])
def test_one_iteration_sums_the_oracles_pixels(dev, cols, rows, level, icp_only, spread):
    f = 0.82 * cols
    c = dict(cols=cols, rows=rows, f=f, cx=0.5 * (cols - 1), cy=0.5 * (rows - 1), voxel=0.01,
             trunc=0.03, buckets=1 << 18, blocks=100000)
    cfg = sys_cfg(c)
    cfg.icp_spread, cfg.icp_only = spread, icp_only
    for i in range(3):
        cfg.icp_iters[i] = 1 if i == level else 0
        cfg.icp_min_count[i] = 1
    g, o, s = B.System(cfg), O.OracleSystem(cfg), synth(c)
    for i in range(2):
        d, rgb, lab = s.render(i)
        g.grab(to_dev(d, dev), to_dev(rgb, dev), to_dev(lab, dev))
        rg, ro = g.result(), o.grab(d, rgb, lab)
        assert rg["tracked"] == ro["tracked"], (rg, ro)  # 160 x 127 alone is lost, on both sides
        assert rg["icp_count"] == ro["icp_count"], (rg, ro)
        assert rg["rgb_count"] == ro["rgb_count"], (rg, ro)
        assert np.abs(rg["pose"] - ro["pose"]).max() < 1e-6
    assert ro["icp_count"] > 0
    assert (ro["rgb_count"] > 0) == (icp_only == 0)
