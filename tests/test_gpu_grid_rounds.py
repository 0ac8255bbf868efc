"""Grid mode is bound by its rounds: on unit-weight mazes their number stays near
the least there can be (the path's length), and small graphs run on few
workgroups, whose launch and barriers are cheap."""
import pytest

import ddp_amd
from oracle import pyoracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,seed", [(64, 1), (100, 2), (300, 3), (512, 1), (512, 2), (1024, 1)])
@pytest.mark.parametrize("K", [64, 1024])
def test_maze_rounds(ctx, side, seed, K):
    hg = ddp_amd.HostGraph.grid_maze(side, side, 300, seed)
    src, dst = hg.reachable_pairs(2, seed)
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=True)
    dg.set_grid(side)
    for s, t in zip(src, dst):
        r = ddp_amd.astar(ctx, dg, int(s), int(t), heur=ddp_amd.H_MANHATTAN, K=K, mode=ddp_amd.MODE_GRID)
        d, _ = pyoracle.dijkstra(hg.off, hg.col, hg.w, int(s), int(t))
        assert r.cost == d[t]
        print(side, seed, K, r.cost, r.stats["iterations"], flush=True)
        assert r.stats["iterations"] <= 1.25 * r.cost + 20  # unit weights: a round a step at least
    dg.close()


@pytest.mark.parametrize("n,deg,blocks", [(1000, 6, 16), (32767, 4, 16), (32769, 4, 64)])
def test_small_graphs_on_few_workgroups(ctx, n, deg, blocks):
    hg = ddp_amd.HostGraph.random(n, deg, 1, 100, n)
    src, dst = hg.reachable_pairs(1, n)
    s, t = int(src[0]), int(dst[0])
    dg = ddp_amd.DeviceGraph(ctx, hg)
    r = ddp_amd.astar(ctx, dg, s, t, heur=ddp_amd.H_ZERO, mode=ddp_amd.MODE_GRID)
    want = pyoracle.dijkstra(hg.off, hg.col, hg.w, s, t)[0][t]
    assert hg.E == n * deg and r.stats["blocks"] == blocks and r.cost == want
    d = ddp_amd.DAStar(ctx, hg, s, t)
    assert d.cost == want
    d.close()
    dg.close()
