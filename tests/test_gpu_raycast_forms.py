"""The raycast's first pass at the sizes and ranges where its own choices can
go wrong, against the oracle, bit for bit (NaN patterns included): images that
do not fill a super-tile or a tile, depth ranges longer than the block cube a
wavefront can name (whose rays the second pass takes), and a camera whose
coordinates cross zero and the powers of two, where neighbouring reads'
coordinates do not round alike."""
import numpy as np
import pytest
import torch

from helpers import B, bits_equal, empty_dev, host, map_cfg, mismatch_report, synth, to_dev
from oracle import binding as O
from test_gpu_map import HALF, _inputs

pytestmark = pytest.mark.gpu


def _cfg(cols, rows, voxel):
    return dict(cols=cols, rows=rows, f=0.82 * cols, cx=(cols - 1) / 2, cy=(rows - 1) / 2,
                voxel=voxel, trunc=3 * voxel, buckets=1 << 16, blocks=60000)


def _both(dev, c, half=False):
    k = B.intrinsics(c["f"], c["f"], c["cx"], c["cy"])
    cfg = map_cfg(c, **(HALF if half else {}))
    gm, om = B.Map(cfg), O.OracleMap(cfg)
    s = synth(c, seed=3)
    for i in (0, 3):
        raw, rgb, n, lab = _inputs(c, s, i)
        pose = B.pose_f(s.pose(i))
        t = [to_dev(a, dev) for a in (raw, rgb, n, lab)]
        B.check(B.lib().sicp_fuse_map_color(gm.h, *[B.image(x) for x in t], 1, B.C.byref(pose),
                                            None, k, None, B.stream_ptr()))
        om.fuse(raw, rgb, n, lab, 1, pose, k)
        torch.cuda.synchronize()
    return gm, om, s, k


def _compare(dev, c, gm, om, zmin, zmax, pose, k):
    v = empty_dev((c["rows"], c["cols"], 4), torch.float32, dev, 0, 7.0)
    n = empty_dev((c["rows"], c["cols"], 4), torch.float32, dev, 0, 7.0)
    zt = [to_dev(z, dev) for z in (zmin, zmax)]
    B.check(B.lib().sicp_raycast(gm.h, B.image(v), B.image(n), B.image(zt[0]), B.image(zt[1]),
                                 B.C.byref(pose), None, k, B.stream_ptr()))
    ov, on = om.raycast(c["cols"], c["rows"], zmin, zmax, pose, k)
    assert bits_equal(host(v), ov), mismatch_report(host(v), ov)
    assert bits_equal(host(n), on), mismatch_report(host(n), on)
    return ov


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("cols,rows", [(8, 8), (75, 61), (513, 65), (65, 129)])
def test_ragged_images(dev, cols, rows, half):
    c = _cfg(cols, rows, 0.01)
    gm, om, s, k = _both(dev, c, half)
    pose = B.pose_f(s.pose(3))
    zc, zr = (cols + 7) // 8, (rows + 7) // 8
    zmin, zmax, _ = om.rendering_blocks(zc, zr, 3.0, 0.1, pose, k)
    ov = _compare(dev, c, gm, om, zmin, zmax, pose, k)
    if cols > 8:
        assert (~np.isnan(ov[..., 0])).mean() > 0.1


def test_long_ranges(dev):
    # 2 mm voxels: 16.3 m is the longest range of one cube; a third of the
    # tiles go beyond it, a third stay well inside, a third are empty
    c = _cfg(96, 72, 0.002)
    gm, om, s, k = _both(dev, c)
    pose = B.pose_f(s.pose(3))
    zr, zc = 9, 12
    zmin = np.full((zr, zc), 0.1, np.float32)
    zmax = np.full((zr, zc), 3.0, np.float32)
    zmax[:, 0::3] = 20.0
    zmin[:, 2::3], zmax[:, 2::3] = 100.0, 0.0
    ov = _compare(dev, c, gm, om, zmin, zmax, pose, k)
    hit = ~np.isnan(ov[..., 0])
    assert hit[:, :8].mean() > 0.1 and hit[:, 8:16].mean() > 0.1 and not hit[:, 16:24].any()


@pytest.mark.parametrize("dx", [0.0, 1e-4, -2.0, 5.12])
def test_shifted_cameras(dev, dx):
    # the same map seen from other places: other roundings of the coordinates
    c = _cfg(160, 120, 0.01)
    gm, om, s, k = _both(dev, c)
    T = s.pose(3).copy()
    T[0, 3] += 0.1 * np.sin(dx)
    T[:3, :3] = T[:3, :3] @ np.array([[np.cos(dx / 50), -np.sin(dx / 50), 0],
                                      [np.sin(dx / 50), np.cos(dx / 50), 0], [0, 0, 1]])
    pose = B.pose_f(T)
    zmin, zmax, _ = om.rendering_blocks(20, 15, 3.0, 0.1, pose, k)
    ov = _compare(dev, c, gm, om, zmin, zmax, pose, k)
    assert (~np.isnan(ov[..., 0])).mean() > 0.2
