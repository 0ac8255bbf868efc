"""Piles of a whole-GPU search that overflow for certain.  A chain of nodes is
expanded one a round; each has an edge to every one of n further nodes, lighter
from round to round, so that every round queues all n again and none of them
is taken before the chain has ended."""
import numpy as np
import pytest

import ddp_amd
from helpers import path_cost
from oracle import pyoracle

pytestmark = pytest.mark.gpu

HEAVY = 100000


def fans(n, rounds, exit_at):
    """Chain 0..rounds - 1 (weight 1), target node `rounds`, the n nodes behind it.
    The target is entered from chain node exit_at (weight 200), or from the
    last of the n nodes (weight 5).  From chain node i the n edges weigh
    HEAVY - 2i, which is above the first window (the mean weight)."""
    chain = np.arange(rounds)
    cols, ws, deg = [], [], []
    far = rounds + 1 + np.arange(n)
    for i in chain:
        c, w = [], []
        if i + 1 < rounds:
            c, w = [i + 1], [1]
        if i == exit_at:
            c, w = c + [rounds], w + [200]
        cols.append(np.concatenate([c, far]))
        ws.append(np.concatenate([w, np.full(n, HEAVY - 2 * i)]))
        deg.append(len(cols[-1]))
    deg = np.concatenate([deg, np.zeros(n, int), [1]])  # target and the n nodes; the last one leads on
    off = np.concatenate([[0], np.cumsum(deg)[:-1]])
    return ddp_amd.HostGraph(off, np.concatenate(cols + [[rounds]]), np.concatenate(ws + [[5]]))


def dijkstra(g, s, t):
    d, _ = pyoracle.dijkstra(*g, s, t)
    return int(d[t]) if d[t] >= 0 else ddp_amd.INF_COST


@pytest.mark.parametrize("mode", [ddp_amd.MODE_AUTO, ddp_amd.MODE_PILES])
def test_dastar_far_and_dormant_do_not_fit_together(ctx, mode):
    """25 rounds of 30,000 entries stay in the far pile, F(t) falls below them and 25
    more go dormant: neither pile is full (1,048,576), but together they are."""
    hg = fans(30000, 50, exit_at=24)
    t = 50
    cur = (hg.off, hg.col, hg.w)
    d = ddp_amd.DAStar(ctx, hg, 0, t, mode=mode)
    assert d.cost == dijkstra(cur, 0, t) == 224
    # the open set is whole: without the short way out the target is reached from the n nodes
    for lines in ([(0, 24, t, 0)], [(1, 30, t, 7)], [(0, 30, t, 0), (0, 49, hg.N - 1, 0)]):
        cur = pyoracle.apply_batch(*cur, lines)[:3]
        cost, _ = d.apply(lines)
        assert cost == dijkstra(cur, 0, t), lines
    d.close()


@pytest.mark.parametrize("exit_at,K", [(24, 64), (-1, 64), (-1, 1024)])
def test_grid_search_larger_than_its_piles(ctx, exit_at, K):
    """1.5M entries, far buffers of two entries a node: rebuilt as often as it takes."""
    hg = fans(30000, 50, exit_at)
    dg = ddp_amd.DeviceGraph(ctx, hg)
    want = dijkstra((hg.off, hg.col, hg.w), 0, 50)
    heap_cap = (2 * hg.N + K - 1) // K  # the least that is no limit
    for kw in (dict(), dict(heap_cap=heap_cap)):
        r = ddp_amd.astar(ctx, dg, 0, 50, heur=ddp_amd.H_ZERO, K=K, mode=ddp_amd.MODE_GRID, **kw)
        assert r.cost == want
        assert path_cost(hg.off, hg.col, hg.w, r.path) == want and r.path[0] == 0 and r.path[-1] == 50
    dg.close()


@pytest.mark.parametrize("mode", [ddp_amd.MODE_AUTO, ddp_amd.MODE_PILES])
def test_dastar_far_pile_overflows(ctx, mode):
    """50 rounds of 30,000 far entries, more than the 1,048,576 the buffer holds."""
    hg = fans(30000, 50, exit_at=-1)
    t = 50
    cur = (hg.off, hg.col, hg.w)
    d = ddp_amd.DAStar(ctx, hg, 0, t, mode=mode)
    assert d.cost == dijkstra(cur, 0, t)
    for how, lines in ((0, [(0, 49, hg.N - 1, 0)]), (1, [(1, 10, t, 9)]), (0, [(0, 10, t, 0), (0, 48, hg.N - 1, 0)])):
        cur = pyoracle.apply_batch(*cur, lines)[:3]
        cost, _ = d.apply(lines, mode=how)
        assert cost == dijkstra(cur, 0, t), lines
    d.close()


def test_dastar_long_session(ctx):
    """Batches that take 30,000 dormant nodes to another value and back leave an
    entry each behind that is current again: 45 rounds of them do not fit the
    1,048,576 entries of the open set, which is rebuilt."""
    n = 30000
    # 0 -> 1 (target, 1000) and 0 -> 2 -> the n nodes (beyond the target), the last of which leads on to 1
    off = np.concatenate([[0, 2, 2], np.full(n, n + 2)])
    hg = ddp_amd.HostGraph(off, np.concatenate([[1, 2], 3 + np.arange(n), [1]]),
                           np.concatenate([[1000, 5], np.full(n, 2000), [3]]))
    d = ddp_amd.DAStar(ctx, hg, 0, 1)
    assert d.cost == 1000
    for k in range(45):
        for w in (6, 5):
            cost, _ = d.apply([(0, 0, 2, 0), (1, 0, 2, w)])
            assert cost == 1000
    cost, _ = d.apply([(0, 0, 1, 0)])  # every dormant node is needed now
    assert cost == 5 + 2000 + 3 and d.path().tolist() == [0, 2, hg.N - 1, 1]
    d.close()


def test_rows_that_grew_past_the_hub_list(ctx):
    """Rows that a session's inserts made long (4.5M edges from 64 nodes, folded into
    the base rows) are more segments in one round than the list sized at opening
    holds: what does not fit is expanded where it was taken."""
    import ctypes

    rng = np.random.default_rng(3)
    n, hubs, each = 100000, 64, 70400
    deg = np.ones(n, np.int64)
    deg[0] = hubs
    off = np.concatenate([[0], np.cumsum(deg)[:-1]])
    col = rng.integers(0, n, deg.sum())
    w = np.full(deg.sum(), 50)
    col[:hubs], w[:hubs] = 1 + np.arange(hubs), 1
    t = n - 1
    hg = ddp_amd.HostGraph(off, col, w)
    d = ddp_amd.DAStar(ctx, hg, 0, t)
    assert d.cost == dijkstra((hg.off, hg.col, hg.w), 0, t)
    u = np.repeat(1 + np.arange(hubs), each)
    v, x = rng.integers(0, n, len(u)), rng.integers(100, 1000, len(u))
    lines = np.ascontiguousarray(np.stack([np.ones(len(u), np.int64), u, v, x], 1).astype(np.int32))
    cost, st = ctypes.c_int32(), ddp_amd._capi.DAStats()
    rc = ddp_amd._capi.lib().ddp_dastar_apply(d._h, lines.ctypes.data_as(ctypes.POINTER(ddp_amd._capi.Update)), len(u),
                                              0, ctypes.byref(cost), ctypes.byref(st))
    assert rc == 0 and st.compacted == 1
    src = np.concatenate([np.repeat(np.arange(n), deg), u])
    order = np.argsort(src, kind="stable")
    cur = (np.searchsorted(src[order], np.arange(n)).astype(np.int32), np.concatenate([hg.col, v])[order].astype(np.int32),
           np.concatenate([hg.w, x])[order].astype(np.uint32))
    want = dijkstra(cur, 0, t)
    assert cost.value == want
    for how in (1, 0):  # over the merged rows: a search from 0, and one resumed at the hubs
        for line in ([(0, 0, 1, 0)], [(1, 0, 1, 1)]):
            cur = pyoracle.apply_batch(*cur, line)[:3]
            c, _ = d.apply(line, mode=how)
            assert c == dijkstra(cur, 0, t)
    d.close()
