"""Host results beside what goes on around a call."""
import threading
import time

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


def test_calls_that_end_during_a_capture(dev):
    """More calls at once than the pool of lent buffers keeps, ending while
    another thread captures a graph in the mode that forbids allocations and
    frees elsewhere: the buffers past the pool are freed then, and the capture
    goes on."""
    threads, rows, cols = 24, 24, 40
    rng = np.random.default_rng(5)
    K = B.intrinsics(30.0, 30.0, 19.5, 11.5)
    pose = B.pose_f(np.eye(4))
    nmap = np.zeros((rows, cols, 4), np.float32)
    nmap[..., 2] = -1.0
    jobs = []
    for t in range(threads):
        v = rng.uniform(-0.02, 0.02, (rows, cols, 4)).astype(np.float32)
        v[..., 2] += np.float32(1.0 + 0.01 * t)
        jobs.append([to_dev(a, dev) for a in (v, v + np.float32(1e-3), nmap, nmap)] +
                    [torch.zeros(B.lib().sicp_icp_partials_size(), dtype=torch.uint8, device=dev),
                     torch.zeros(29, dtype=torch.float32, device=dev)])
    streams = [torch.cuda.Stream() for _ in range(threads)]
    capturing = torch.cuda.Stream()
    a, b = torch.randn(4096, 4096, device=dev), torch.empty(4096, 4096, device=dev)
    torch.mm(a, a, out=b)
    torch.cuda.synchronize()
    # every call waits for this work (about half a second), so all of them hold
    # a buffer when the capture begins
    with torch.cuda.stream(streams[0]):
        for _ in range(400):
            torch.mm(a, a, out=b)
        done = torch.cuda.Event()
        done.record()
    for st in streams[1:]:
        st.wait_event(done)
    codes, counts = [[None, None] for _ in range(threads)], np.zeros((threads, 2), np.float32)
    again = threading.Event()

    def run(t):
        v, vl, n, nl, partials, sums = jobs[t]
        for k in range(2):
            hs = np.zeros(29, np.float32)
            codes[t][k] = B.lib().sicp_icp_step(
                B.image(v), B.image(vl), B.image(n), B.image(nl), B.C.byref(pose),
                B.C.byref(pose), K, partials.data_ptr(), sums.data_ptr(),
                hs.ctypes.data_as(B.C.c_void_p), None, None, None, B.stream_ptr(streams[t]))
            counts[t, k] = hs[28]
            again.wait()

    ts = [threading.Thread(target=run, args=(t,)) for t in range(threads)]
    for th in ts:
        th.start()
    time.sleep(0.1)
    hip, graph, status, st = B.lib(), B.C.c_void_p(), B.C.c_int(-1), B.stream_ptr(capturing)
    early = done.query()
    began = hip.hipStreamBeginCapture(st, 0)  # hipStreamCaptureModeGlobal
    for _ in range(1000):
        if all(c[0] is not None for c in codes):
            break
        time.sleep(0.01)
    hip.hipStreamIsCapturing(st, B.C.byref(status))
    ended = hip.hipStreamEndCapture(st, B.C.byref(graph))
    if graph:
        hip.hipGraphDestroy(graph)
    again.set()
    for th in ts:
        th.join()
    hip.hipGetLastError()
    torch.cuda.synchronize()
    assert not early, "the calls did not outlast the capture's begin"
    assert (began, status.value, ended) == (0, 1, 0)
    assert codes == [[0, 0]] * threads
    assert (counts > 0).all()
