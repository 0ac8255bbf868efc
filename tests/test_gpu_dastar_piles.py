"""DA* on the whole-GPU piles at the sizes where its paths change: a near ring
that overflows and is rebuilt, an open set that was limited by heap_cap, batches
of one line and of only inserts or deletes, recomputes between repairs."""
import numpy as np
import pytest

import ddp_amd
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def dijkstra(g, s, t):
    d, _ = pyoracle.dijkstra(*g, s, t)
    return int(d[t]) if d[t] >= 0 else ddp_amd.INF_COST


def sweeps(n, k):
    """Node 0 with k parallel edges to each of n nodes, in k sweeps of falling
    weight (most of them improve their target when they are scanned), and each
    node with two more edges."""
    rng = np.random.default_rng(n + k)
    off = np.full(n, n * k, np.int64)
    off[0] = 0
    off[1:] += 2 * np.arange(n - 1)
    col = np.concatenate([np.tile(np.arange(n), k), rng.integers(0, n, 2 * (n - 1))])
    w = np.concatenate([np.repeat(20 * np.arange(k, 0, -1), n), rng.integers(1, 400, 2 * (n - 1))])
    return ddp_amd.HostGraph(off, col, w)


@pytest.mark.parametrize("mode", [ddp_amd.MODE_AUTO, ddp_amd.MODE_PILES])
def test_dastar_rebuild(ctx, mode):
    """2M edges from one node: far more near entries in one round than the ring
    holds (65,536 for 40,000 nodes)."""
    hg = sweeps(40000, 50)
    t = hg.N - 1
    d = ddp_amd.DAStar(ctx, hg, 0, t, mode=mode)
    cur = (hg.off, hg.col, hg.w)
    assert d.cost == dijkstra(cur, 0, t)
    for k in range(3):
        lines = [(0, 0, t, 0)] * 7 + [(0, int(v), int(hg.col[hg.off[v]]), 0) for v in range(1 + k, 200, 3)]
        cur = pyoracle.apply_batch(*cur, lines)[:3]
        cost, _ = d.apply(lines, mode=ddp_amd.DAStar.REPAIR if k != 1 else ddp_amd.DAStar.RECOMPUTE)
        assert cost == dijkstra(cur, 0, t)
    d.close()


def test_dastar_open_set_limit(ctx):
    """An open set limited by heap_cap ends with DDP_ERR_OVERFLOW, as its queues did."""
    hg = sweeps(30000, 1)
    with pytest.raises(ddp_amd.DDPError) as e:
        ddp_amd.DAStar(ctx, hg, 0, hg.N - 1, K=64, heap_cap=32)
    assert e.value.code == 4


@pytest.mark.parametrize("n,deg", [(50, 3), (3000, 5), (200000, 4)])
def test_dastar_batch_kinds(ctx, n, deg):
    hg = ddp_amd.HostGraph.random(n, deg, 1, 100, n)
    src, dst = hg.reachable_pairs(1, n)
    s, t = int(src[0]), int(dst[0])
    rng = np.random.default_rng(n)
    off = hg.offsets_full()
    d = ddp_amd.DAStar(ctx, hg, s, t, K=1024)
    cur = (hg.off, hg.col, hg.w)
    for k in range(10):
        path = [int(x) for x in d.path()] if d.cost != ddp_amd.INF_COST else []
        dels = [(0, a, b, 0) for a, b in zip(path[:-1], path[1:])][:1 + k % 3]
        u = rng.integers(0, n, 1 if k == 0 else 40)
        dels += [(0, int(a), int(hg.col[off[a]]), 0) for a in u]
        ins = [(1, int(a), int(b), int(w)) for a, b, w in zip(u, rng.integers(0, n, 40), rng.integers(1, 100, 40))]
        lines = (ins[:1], dels, ins, dels[:1], dels + ins)[k % 5]
        cur = pyoracle.apply_batch(*cur, lines)[:3]
        cost, st = d.apply(lines, mode=ddp_amd.DAStar.RECOMPUTE if k in (4, 7) else ddp_amd.DAStar.REPAIR)
        assert cost == dijkstra(cur, s, t), k
        assert st["inserts"] + st["deletes"] == len(lines)
    d.close()
