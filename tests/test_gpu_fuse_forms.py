"""The fusion's packed pixel record keeps "has a normal" in the depth's sign
where every valid depth is positive, and reads the normal map itself where
depth_min is not above zero: both, with and without labels and in the half
form, on an odd image size, against the oracle bit for bit."""
import pytest

from helpers import B, CFG_SMALL, map_cfg
from oracle import binding as O
from test_gpu_map import HALF, _compare_maps, _fuse_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth_min", [0.1, 0.0, -1.0])
@pytest.mark.parametrize("labels", [True, False])
@pytest.mark.parametrize("half", [False, True])
def test_pixel_record_forms(dev, depth_min, labels, half):
    c = dict(CFG_SMALL, cols=161, rows=119, f=131.25, cx=80.0, cy=59.0)
    cfg = map_cfg(c, depth_min=depth_min, **(HALF if half else {}))
    gm, om = B.Map(cfg), O.OracleMap(cfg)
    _fuse_both(dev, c, [1, 4, 7], gm, om, labels=labels)
    assert _compare_maps(gm, om) > 100
