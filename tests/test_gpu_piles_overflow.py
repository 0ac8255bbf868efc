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
