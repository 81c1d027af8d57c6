"""Mesh calls on one map from several threads at once: one call has the scratch
kept with the map, the others allocate their own, and each gives the mesh of a
call alone, word for word."""
import threading

import pytest
import torch

from helpers import B, CFG_SMALL, map_cfg
from oracle import binding as O
from test_gpu_map import _fuse_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threads", [4])
def test_mesh_from_several_threads(dev, threads):
    cfg = map_cfg(CFG_SMALL)
    gm = B.Map(cfg)
    _fuse_both(dev, CFG_SMALL, [0, 2], gm, O.OracleMap(cfg))
    v, n, col, total = gm.mesh(1 << 18)
    torch.cuda.synchronize()
    assert 1000 < total <= 1 << 18
    bad = []
    streams = [torch.cuda.Stream() for _ in range(threads)]

    def run(k):
        with torch.cuda.stream(streams[k]):
            for _ in range(5):
                a = gm.mesh(1 << 18)
                streams[k].synchronize()
                if a[3] != total or not (torch.equal(a[0], v) and torch.equal(a[2], col) and
                                         torch.equal(torch.nan_to_num(a[1], 9.0),
                                                     torch.nan_to_num(n, 9.0))):
                    bad.append(k)

    ts = [threading.Thread(target=run, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
