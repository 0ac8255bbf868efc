"""Claims of a burst do not hold up the searches that run beside them."""
import numpy as np
import pytest

import ddp_amd

pytestmark = pytest.mark.gpu


def test_more_slots_than_arrivals_need(ctx):
    """Thousands of short queries on twice the slots that keep up with their
    arrival: the slowest searches take no more than twice as long as with half
    the slots (they took four times as long beside slots that fought over claims)."""
    hg = ddp_amd.HostGraph.geometric(200000, 10, 100000, 1)
    src, dst = hg.geo_pairs(8192, 2000, 100000, 1)
    dg = ddp_amd.DeviceGraph(ctx, hg, reorder=True)
    n = len(src)
    slow, costs = {}, []
    for slots in (256, 512):
        sv = ddp_amd.Server(ctx, dg, heur=ddp_amd.H_EUCLID, block=512, slots=slots, idle_ms=200)
        assert sv.info()["slots"] == slots
        p = []
        for k in range(4):
            res = sv.replay(np.zeros(n), np.zeros(n, np.int32), src, dst, [None] * n)
            assert all(r["status"] == 0 for r in res)
            p.append(np.percentile([r["device_ms"] for r in res], 99.9))
        slow[slots] = sorted(p[1:])[1]
        costs.append([r["cost"] for r in res])
        sv.close()
    print(slow, flush=True)
    assert costs[0] == costs[1]
    assert slow[512] < 2 * slow[256]
    dg.close()
