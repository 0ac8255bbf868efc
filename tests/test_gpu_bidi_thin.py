"""Thin rounds of the bidirectional engine (short rows, few entries a round)
and its two-lane path walk, at the sizes where they can go wrong: rows just
below, at and above the row limit, hub rows among short ones, more and fewer
entries a round than a direction's lanes, every block width that has them, and
paths longer than the far piles that the walk borrows.  Weights are drawn so
that costs are exact integers: costs equal the oracle's, no tolerance."""
import numpy as np
import pytest

import ddp_amd
from helpers import path_cost
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def layered(rng, width, layers, deg, hub):
    """layers x width nodes; each has deg edges into the next layer (one node
    per layer has `hub`), two back; node 0 leads in, the last node leads out."""
    N = layers * width + 2
    rows = [[] for _ in range(N)]
    rows[0] = [1 + i for i in range(width)]
    for a in range(layers):
        for i in range(width):
            u = 1 + a * width + i
            if a + 1 < layers:
                k = hub if i == a % width else deg
                rows[u] += (1 + (a + 1) * width + rng.integers(0, width, k)).tolist()
            else:
                rows[u].append(N - 1)
            if a:
                rows[u] += (1 + (a - 1) * width + rng.integers(0, width, 2)).tolist()
    off = np.zeros(N, np.int32)
    off[1:] = np.cumsum([len(r) for r in rows])[:-1]
    col = np.concatenate([np.asarray(r, np.int32) for r in rows if r]).astype(np.int32)
    w = rng.integers(1, 40, len(col)).astype(np.uint32)
    return off, col, w


def want(hg, src, dst):
    out = []
    for s, t in zip(src, dst):
        d, _ = pyoracle.dijkstra(hg.off, hg.col, hg.w, int(s), int(t))
        out.append(int(d[t]) if d[t] >= 0 else ddp_amd.INF_COST)
    return np.asarray(out, np.int64)


def check(hg, src, dst, costs, paths):
    assert np.array_equal(costs, want(hg, src, dst))
    for i, p in enumerate(paths):
        if costs[i] == ddp_amd.INF_COST:
            assert len(p) == 0
        else:
            assert p[0] == src[i] and p[-1] == dst[i]
            assert path_cost(hg.off, hg.col, hg.w, p) == costs[i]


# deg: the row limit is 8 and two back edges are added, so 5, 6, 7 are rows of
# 7, 8 and 9; width: entries a round around a direction's 64 (256 lanes) and 128
@pytest.mark.parametrize("block", [256, 512])
@pytest.mark.parametrize("deg,hub", [(1, 1), (5, 5), (6, 6), (7, 7), (4, 60), (6, 700)])
@pytest.mark.parametrize("width", [3, 64, 130])
def test_thin_rows_and_widths(ctx, block, deg, hub, width):
    rng = np.random.default_rng(1000 * deg + 10 * width + block)
    hg = ddp_amd.HostGraph(*layered(rng, width, 24, deg, hub))
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=True)
    print("thin", block, deg, hub, width, flush=True)
    src = np.concatenate([[0, 0, hg.N - 1], rng.integers(0, hg.N, 21)]).astype(np.int32)
    dst = np.concatenate([[hg.N - 1, 0, 0], rng.integers(0, hg.N, 21)]).astype(np.int32)
    costs, paths, st = ddp_amd.astar_batch(ctx, dg, src, dst, heur=ddp_amd.H_ZERO, block=block, path_cap=hg.N + 1,
                                           engine=ddp_amd.ENGINE_BIDI, slots=8)
    assert st["errors"] == 0
    check(hg, src, dst, costs, paths)
    dg.close()


@pytest.mark.parametrize("K", [256, 512])
@pytest.mark.parametrize("W,H", [(64, 64), (3, 5000), (701, 13)])
def test_thin_maze_paths(ctx, K, W, H):
    """Manhattan mazes, among them corridors of thousands of hops: the walk's
    chains are as long as a search can make them, with and without room in
    the smallest piles a caller may ask for."""
    hg = ddp_amd.HostGraph.grid_maze(W, H, 200, 5)
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=True)
    dg.set_grid(W)
    src, dst = [0, hg.N - 1, 7], [hg.N - 1, 0, 7]
    ref = want(hg, src, dst)
    print("thin maze", K, W, H, flush=True)
    for s, t, c in zip(src, dst, ref):
        r = ddp_amd.astar(ctx, dg, s, t, heur=ddp_amd.H_MANHATTAN, K=K, mode=ddp_amd.MODE_BIDI)
        assert r.cost == c and r.path[0] == s and r.path[-1] == t
        assert path_cost(hg.off, hg.col, hg.w, r.path) == c
    for cap in (0, 1024):  # default scratch and small piles
        costs, paths, st = ddp_amd.astar_batch(ctx, dg, src, dst, heur=ddp_amd.H_MANHATTAN, block=K, heap_cap=cap,
                                               path_cap=hg.N, engine=ddp_amd.ENGINE_BIDI)
        assert st["errors"] == 0
        check(hg, src, dst, costs, paths)
    dg.close()
