"""Host results beside what goes on around a call."""
import numpy as np
import pytest
import torch

from helpers import B, CFG_SMALL, sys_cfg, synth, to_dev

pytestmark = pytest.mark.gpu


def test_frame_result_after_another_calls_error(dev):
    """sicp_system_last_result answers for its own work alone: a HIP call that
    failed before in the thread (here: a device that does not exist) does not
    make it fail."""
    g = B.System(sys_cfg(CFG_SMALL))
    s = synth(CFG_SMALL)
    for i in range(2):
        g.grab(*[to_dev(a, dev) for a in s.render(i)])
    torch.cuda.synchronize()
    want = g.result()
    hip = B.lib()  # its HIP runtime, whose last error is the thread's
    try:
        assert hip.hipSetDevice(1 << 20) != 0
        got = g.result()
    finally:
        hip.hipGetLastError()
    assert np.array_equal(got.pop("pose"), want.pop("pose"))
    assert got == want
