"""Fusion with every label a mask can hold (0..255), against the oracle bit for
bit. A label's colour is (palette x label) % 255 in wrapping 32-bit arithmetic
(FuseMap.cu:18,570-572), negative in the first channel for half of the labels
from 65 on, and narrowed to a byte where it is stored: nothing of it may reach
the record's other bytes."""
import numpy as np
import pytest

from helpers import B, CFG_SMALL, K, map_cfg, synth, to_dev
from oracle import binding as O
from test_gpu_map import HALF, _compare_maps, _inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("low,high", [(0, 256), (60, 82), (128, 200)])
def test_every_label_bit_exact(dev, half, low, high):
    c = dict(CFG_SMALL, cols=161, rows=119, f=131.25, cx=80.0, cy=59.0)
    cfg = map_cfg(c, **(HALF if half else {}))
    gm, om = B.Map(cfg), O.OracleMap(cfg)
    s = synth(c)
    y, x = np.mgrid[0:c["rows"], 0:c["cols"]]
    tile = (y // 6) * 27 + x // 6
    for k in range(9):
        raw, rgb, n, _ = _inputs(c, s, k % 3)
        # three labels a tile in turn, so that labels are seen again, replaced
        # as the second one and swapped; a tenth of the pixels background
        lab = (low + (tile * 5 + (k // 2) % 3) % (high - low)).astype(np.uint8)
        lab[(x * 7 + y * 3 + k) % 10 == 0] = 0
        pose = B.pose_f(s.pose(k % 3))
        t = [to_dev(a, dev) for a in (raw, rgb, n, lab)]
        B.check(B.lib().sicp_fuse_map_color(gm.h, *[B.image(v) for v in t], 1, B.C.byref(pose),
                                            None, K(c), None, B.stream_ptr()))
        om.fuse(raw, rgb, n, lab, 1, pose, K(c))
    assert _compare_maps(gm, om) > 100
    sem = om.export()["sem"]
    assert len(np.unique(sem["label"])) > (high - low) // 2
