"""The neighbour label pass far from the origin, where the rounding of world
coordinates moves the probes by whole voxels (its staged label words then do
not hold every probe), against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

from helpers import B, CFG_SMALL, K, map_cfg, synth, to_dev
from oracle import binding as O
from test_gpu_map import _compare_maps, _inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0.0, -3.0e3, 2.0e4, 7.0e4])
def test_unify_at_large_coordinates(dev, shift):
    # 1 cm voxels: 7e4 m is voxel 7e6 of the keys' 8.4e6
    c = CFG_SMALL
    cfg = map_cfg(c, unify_labels=1)
    gm, om = B.Map(cfg), O.OracleMap(cfg)
    s = synth(c, seed=5)
    for i in (0, 2, 4):
        raw, rgb, n, lab = _inputs(c, s, i)
        T = s.pose(i).copy()
        T[0, 3] += shift
        T[2, 3] -= 0.5 * shift
        pose = B.pose_f(T)
        t = [to_dev(a, dev) for a in (raw, rgb, n, lab)]
        B.check(B.lib().sicp_fuse_map_color(gm.h, *[B.image(x) for x in t], 1, B.C.byref(pose),
                                            None, K(c), None, B.stream_ptr()))
        om.fuse(raw, rgb, n, lab, 1, pose, K(c))
        torch.cuda.synchronize()
    n = _compare_maps(gm, om)
    assert n > 100
