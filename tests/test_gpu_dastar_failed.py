"""A DA* batch whose search fails (an open set limited by heap_cap) is part of
the graph, and the session answers exactly or with an error afterwards."""
import numpy as np
import pytest

import ddp_amd
from oracle import pyoracle

pytestmark = pytest.mark.gpu

LEAVES = 5000


def fan():
    """0 -> 1 (the target) directly, and 0 -> 2 -> LEAVES nodes, one of which leads
    on to 1: without the direct edge a search has all leaves open at once."""
    n = 3 + LEAVES
    off = np.full(n, 2 + LEAVES, np.int32)
    off[:3] = 0, 2, 2
    last = n - 1 - LEAVES // 3
    off[last + 1:] += 1
    col = np.concatenate([[1, 2], np.arange(3, n), [1]])
    w = np.concatenate([[1, 5], np.full(LEAVES, 1000), [1]])
    return ddp_amd.HostGraph(off, col, w)


@pytest.mark.parametrize("mode", [ddp_amd.DAStar.REPAIR, ddp_amd.DAStar.RECOMPUTE])
def test_session_after_overflow(ctx, mode):
    hg = fan()
    d = ddp_amd.DAStar(ctx, hg, 0, 1, K=64, heap_cap=32)  # 2,048 entries
    assert d.cost == 1
    cur = (hg.off, hg.col, hg.w)
    failing = [(0, 0, 1, 0), (1, 0, 7, 3000), (1, 0, 9, 3000)]
    cur = pyoracle.apply_batch(*cur, failing)[:3]
    with pytest.raises(ddp_amd.DDPError) as e:
        d.apply(failing, mode=mode)
    assert e.value.code == 4
    with pytest.raises(ddp_amd.DDPError) as e:
        d.path()
    assert e.value.code == 8

    def same_graph():
        g = d.graph()
        assert [x.tolist() for x in (g.off, g.col, g.w)] == [np.asarray(x).tolist() for x in cur]

    same_graph()
    dist, _ = pyoracle.dijkstra(*cur, 0, 1)
    assert dist[1] == 1006
    for lines in ([(0, 0, 8, 0)], []):  # still too many open nodes: an error again, never another cost
        try:
            cost, _ = d.apply(lines, mode=mode)
            assert cost == 1006
        except ddp_amd.DDPError as e:
            assert e.code == 4
    lines = [(1, 0, 1, 4)]
    cur = pyoracle.apply_batch(*cur, lines)[:3]
    cost, st = d.apply(lines, mode=mode)
    assert cost == 4 and d.path().tolist() == [0, 1]
    same_graph()
    lines = [(1, 0, 1, 3), (0, 2, 3, 0)]
    cur = pyoracle.apply_batch(*cur, lines)[:3]
    cost, st = d.apply(lines, mode=mode)
    assert cost == 3 and st["deletes_effective"] == 1
    same_graph()
    d.close()
