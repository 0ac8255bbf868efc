"""Grid mode (piles over the whole GPU) at the sizes where its paths change:
rows around the length at which they are cut into segments and hubs that span
the grid, windows from one entry to whole graphs, both launch widths, the
limits it reports.  Costs against Dijkstra, paths edge by edge."""
import numpy as np
import pytest

import ddp_amd
from helpers import path_cost
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def hub_graph(deg, n, seed):
    """Hub 0 with deg edges (parallel ones of other weights among them), every
    node with two more edges, some edges deleted."""
    rng = np.random.default_rng(seed)
    degree = np.full(n, 2)
    degree[0] = deg
    off = np.concatenate([[0], np.cumsum(degree)[:-1]]).astype(np.int32)
    col = rng.integers(0, n, degree.sum()).astype(np.int32)
    col[rng.integers(0, len(col), len(col) // 50)] = -1
    return ddp_amd.HostGraph(off, col, rng.integers(1, 1000, len(col)))


def check(ctx, hg, s, targets, K, heur=ddp_amd.H_ZERO, dg=None):
    d, _ = pyoracle.dijkstra(hg.off, hg.col, hg.w, s)
    dg = dg or ddp_amd.DeviceGraph(ctx, hg)
    for t in targets:
        r = ddp_amd.astar(ctx, dg, s, int(t), heur=heur, K=K, mode=ddp_amd.MODE_GRID)
        assert r.cost == (int(d[t]) if d[t] >= 0 else ddp_amd.INF_COST), (K, s, t)
        if r.found:
            assert r.path[0] == s and r.path[-1] == t
            assert path_cost(hg.off, hg.col, hg.w, r.path) == r.cost
        else:
            assert len(r.path) == 0
    return dg


@pytest.mark.parametrize("deg", [63, 64, 65, 128, 129, 5000, 300001])
@pytest.mark.parametrize("K", [1, 1024, 65536])
def test_grid_hub_rows(ctx, deg, K):
    hg = hub_graph(deg, 4000, deg)
    s = next(int(u) for u in range(1, hg.N) if hg.col[hg.off[u]] >= 0)
    check(ctx, hg, 0, [0, 17, 3999], K).close()
    check(ctx, hg, s, [0, s, 2000], K).close()


@pytest.mark.parametrize("scale", [17, 18])  # 64 workgroups, then (4.2M edges) one per CU
def test_grid_launch_widths(ctx, scale):
    hg = ddp_amd.HostGraph.rmat(scale, 16 << scale, 0.57, 0.19, 0.19, 1, 1000, scale)
    src, dst = hg.hub_pairs(2, 3)
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=True, reorder=True)
    for s, t in zip(src, dst):
        check(ctx, hg, int(s), [t, 0], 4096, dg=dg)
    r = ddp_amd.astar(ctx, dg, int(src[0]), int(dst[0]), heur=ddp_amd.H_ZERO, K=64, mode=ddp_amd.MODE_GRID)
    assert r.stats["blocks"] == (64 if scale == 17 else ctx.device_info()["compute_units"])
    dg.close()


def test_grid_limits(ctx):
    """Piles that are too small and iteration limits end with the errors they had
    (DDP_ERR_OVERFLOW, DDP_ERR_TIMEOUT)."""
    hg = hub_graph(20000, 30000, 1)
    dg = ddp_amd.DeviceGraph(ctx, hg)
    for kw, code in ((dict(heap_cap=1, lds_cap=1), 4), (dict(max_iters=1), 7)):
        with pytest.raises(ddp_amd.DDPError) as e:
            ddp_amd.astar(ctx, dg, 0, 29999, heur=ddp_amd.H_ZERO, K=64, mode=ddp_amd.MODE_GRID, **kw)
        assert e.value.code == code
    check(ctx, hg, 0, [29999], 64, dg=dg).close()  # and the next search starts clean
