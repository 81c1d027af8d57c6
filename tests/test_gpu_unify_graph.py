"""The neighbour label pass in the graph form of a frame and of a batch's round:
replays see the same blocks in the pass's snapshot as eager launches do, also
where blocks leave the view and their neighbours stay in it, so the maps are the
same bytes."""
import numpy as np
import pytest
import torch

from helpers import B, CFG_SMALL, sys_cfg, synth, to_dev
from test_gpu_batched import _map_state

pytestmark = pytest.mark.gpu

FRAMES = 40


def _config():
    return sys_cfg(CFG_SMALL, unify_labels=1)


def _frames(dev, seed):
    s = synth(CFG_SMALL, seed=seed)
    return [[to_dev(a, dev) for a in s.render(i)] for i in range(FRAMES)]


def _same(a, b):
    (na, da), (nb, db) = _map_state(a), _map_state(b)
    assert na == nb and na > 500
    for f in da["sem"].dtype.names:
        diff = np.count_nonzero(da["sem"][f] != db["sem"][f])
        assert diff == 0, (f, diff)
    for f in ("table", "excess", "blocks", "geom"):
        assert np.array_equal(da[f].view(np.uint8), db[f].view(np.uint8)), f
    assert len(np.unique(da["sem"]["label"])) > 2


def test_graph_replays_equal_eager_launches(dev):
    eager, graph = B.System(_config()), B.System(_config())
    visible = []
    for t in _frames(dev, 0):
        eager.grab(*t)
        graph.grab_staged(*t, use_graph=True)
        re, rg = eager.result(), graph.result()
        assert re["tracked"] == rg["tracked"] == 1
        assert np.array_equal(re["pose"], rg["pose"])
        visible.append((re["visible_blocks"], re["allocated_blocks"]))
    assert visible[-1][0] < 0.9 * visible[-1][1]  # blocks did leave the view
    _same(eager, graph)


@pytest.mark.parametrize("shared", [True, False])
def test_batch_rounds_equal_eager_launches(dev, shared):
    frames = [_frames(dev, k) for k in (0, 1)]
    eager, graph = ([B.System(_config()) for _ in frames] for _ in range(2))
    batch = B.Batch(graph)
    batch.set_shared_tracking(shared)
    for i in range(FRAMES):
        for g, f in zip(eager, frames):
            g.grab(*f[i])
        batch.grab_staged([f[i] for f in frames], True)
    torch.cuda.synchronize()
    for a, b in zip(eager, graph):
        _same(a, b)
    batch.close()
