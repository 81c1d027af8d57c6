"""Host results of the step entry points come through lent pinned buffers: from
more threads at once than the pool keeps idle, also while the idle ones are
freed (a system destroyed), each call gets its own sums: those of its device
buffer, which hold the same words."""
import threading

import numpy as np
import pytest
import torch

from helpers import B, CFG_SMALL, sys_cfg, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threads,release", [(1, False), (24, False), (4, True)])
def test_concurrent_calls_get_their_own_sums(dev, threads, release):
    rng = np.random.default_rng(5)
    rows, cols = 24, 40
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
    torch.cuda.synchronize()
    seen, bad = [], []

    def run(t):
        v, vl, n, nl, partials, sums = jobs[t]
        with torch.cuda.stream(streams[t]):
            for _ in range(20):
                hs = np.zeros(29, np.float32)
                B.check(B.lib().sicp_icp_step(
                    B.image(v), B.image(vl), B.image(n), B.image(nl), B.C.byref(pose),
                    B.C.byref(pose), K, partials.data_ptr(), sums.data_ptr(),
                    hs.ctypes.data_as(B.C.c_void_p), None, None, None, B.stream_ptr()))
                seen.append(hs[28])
                if not np.array_equal(hs, sums.cpu().numpy()):
                    bad.append(t)

    ts = [threading.Thread(target=run, args=(t,)) for t in range(threads)]
    for th in ts:
        th.start()
    if release:
        B.System(sys_cfg(CFG_SMALL)).close()
    for th in ts:
        th.join()
    assert not bad
    assert len(seen) == 20 * threads and min(seen) > 0
