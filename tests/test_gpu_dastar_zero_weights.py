"""Zero-weight edges that enter a DA* session by updates, and become base rows
when the log is folded in: costs stay exact and the parents lead back to s."""
import numpy as np
import pytest

import ddp_amd
from helpers import path_cost
from oracle import pyoracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,deg,seed", [(60, 3, 1), (3000, 4, 2), (40000, 4, 3)])
def test_zero_weight_inserts_compacted(ctx, n, deg, seed):
    hg = ddp_amd.HostGraph.random(n, deg, 1, 4, seed)
    src, dst = hg.reachable_pairs(1, seed)
    s, t = int(src[0]), int(dst[0])
    rng = np.random.default_rng(seed)
    d = ddp_amd.DAStar(ctx, hg, s, t)
    cur = (hg.off, hg.col, hg.w)

    def step(lines, mode):
        nonlocal cur
        cur = pyoracle.apply_batch(*cur, lines)[:3]
        cost, _ = d.apply(lines, mode=mode)
        dist, _ = pyoracle.dijkstra(*cur, s, t)
        assert cost == (int(dist[t]) if dist[t] >= 0 else ddp_amd.INF_COST)
        if cost != ddp_amd.INF_COST:
            p = d.path()
            assert p[0] == s and p[-1] == t and path_cost(*cur, p) == cost

    for k in range(8):
        # rings of zero weight through random nodes, both ways round
        ring = rng.permutation(n)[:n // 10]
        lines = [(1, int(a), int(b), 0) for a, b in zip(ring, np.roll(ring, -1))]
        lines += [(1, int(b), int(a), 0) for a, b in zip(ring, np.roll(ring, -1))]
        path = [int(x) for x in d.path()] if d.cost != ddp_amd.INF_COST else []
        lines += [(0, a, b, 0) for a, b in list(zip(path[:-1], path[1:]))[::2]]
        step(lines, ddp_amd.DAStar.REPAIR if k % 3 else ddp_amd.DAStar.RECOMPUTE)
        if k % 2 == 0:
            d.compact()
    d.close()
