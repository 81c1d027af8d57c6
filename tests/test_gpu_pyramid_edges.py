"""The pyramid kernels' forms for wavefronts away from the image's edges, and
the filter's for depths near each other, against the oracle bit for bit: images
around one 64x4 tile, pitched, and depths whose differences lie on both sides
of the near form's bound (6.5 m) in the same tile, or everywhere; a scale that
makes every depth infinite. The two forms compute the same float operations, so
no difference is allowed."""
import numpy as np
import pytest
import torch

from helpers import B, bits_equal, empty_dev, host, mismatch_report, to_dev
from oracle import binding as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,rows", [(8, 8), (63, 5), (64, 9), (66, 12), (129, 33), (200, 70)])
@pytest.mark.parametrize("far,scale", [(0.0, 1000.0), (0.01, 1000.0), (1.0, 1000.0),
                                       (0.2, 5000.0), (0.2, 1e-36)])
def test_filter_forms(dev, cols, rows, far, scale):
    rng = np.random.default_rng(cols * rows)
    d = rng.integers(400, 6900, (rows, cols)).astype(np.uint16)   # within 6.5 m at 1000
    wide = rng.integers(0, 65536, (rows, cols)).astype(np.uint16)
    d = np.where(rng.random((rows, cols)) < far, wide, d)
    dt = to_dev(d, dev, 3)
    raw = empty_dev((rows, cols), torch.float32, dev, 3)
    filt = empty_dev((rows, cols), torch.float32, dev, 3)
    B.check(B.lib().sicp_filter_depth(B.image(dt), B.image(raw), B.image(filt), scale, 60.0,
                                      B.stream_ptr()))
    oraw, ofilt = O.filter_depth(d, scale, 60.0)
    assert bits_equal(host(raw), oraw), mismatch_report(host(raw), oraw)
    assert bits_equal(host(filt), ofilt), mismatch_report(host(filt), ofilt)


@pytest.mark.parametrize("cols,rows", [(8, 8), (129, 9), (131, 22), (260, 39), (400, 70)])
@pytest.mark.parametrize("holes", [0.0, 0.5, 1.0])
def test_pyrdown_and_derivative_forms(dev, cols, rows, holes):
    rng = np.random.default_rng(cols * rows)
    src = rng.uniform(0.2, 9.0, (rows, cols)).astype(np.float32)
    src[rng.random((rows, cols)) < holes] = np.nan
    dst = empty_dev((rows // 2, cols // 2), torch.float32, dev, 2)
    B.check(B.lib().sicp_pyrdown_gauss_f32(B.image(to_dev(src, dev, 1)), B.image(dst),
                                           B.stream_ptr()))
    ref = O.pyrdown_f32(src)
    assert bits_equal(host(dst), ref), mismatch_report(host(dst), ref)
    gray = rng.integers(0, 256, (rows, cols)).astype(np.uint8)
    g = to_dev(gray, dev, 1)
    gd = empty_dev((rows // 2, cols // 2), torch.uint8, dev, 2)
    B.check(B.lib().sicp_pyrdown_gauss_u8(B.image(g), B.image(gd), B.stream_ptr()))
    assert np.array_equal(host(gd), O.pyrdown_u8(gray))
    dx = empty_dev((rows, cols), torch.int16, dev, 2)
    dy = empty_dev((rows, cols), torch.int16, dev, 2)
    B.check(B.lib().sicp_compute_derivative_image(B.image(g), B.image(dx), B.image(dy),
                                                  B.stream_ptr()))
    odx, ody = O.derivative_image(gray)
    assert np.array_equal(host(dx), odx) and np.array_equal(host(dy), ody)
