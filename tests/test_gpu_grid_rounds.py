"""Grid mode is bound by its rounds: on unit-weight mazes their number stays near
the least there can be (the path's length)."""
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
