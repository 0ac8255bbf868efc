"""Requests that had kernels of their own (grid mode) go several times round the
ring before a serve launch sees any of them: it passes over all of them and runs
each later request once."""
import numpy as np
import pytest

import ddp_amd
from oracle import pyoracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("engine", [ddp_amd.ENGINE_PILES, ddp_amd.ENGINE_BIDI])
def test_ring_wraps_between_launches(ctx, engine):
    hg = ddp_amd.HostGraph.random(1500, 5, 1, 100, 31)
    upd = hg.gen_updates(12, 20, 20, 1, 100, 32)
    versions = [(hg.off, hg.col, hg.w)]
    for b in upd.batches:
        versions.append(pyoracle.apply_batch(*versions[-1], b)[:3])
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=True)
    rng = np.random.default_rng(33)
    sv = ddp_amd.Server(ctx, dg, heur=ddp_amd.H_ZERO, ring=64, slots=16, block=256, engine=engine, grid_k=256,
                        idle_ms=5)
    got, plan, tag, v = {}, {}, 0, 0

    def query():
        nonlocal tag
        s, t = int(rng.integers(0, 30)), int(rng.integers(0, hg.N))
        assert sv.submit_query(s, t, tag) == 0
        plan[tag] = (v, s, t)
        tag += 1

    def update():
        nonlocal tag, v
        assert sv.submit_update(upd.batches[v], tag) == 0
        v += 1
        plan[tag] = (v, None, None)
        tag += 1

    def settle():
        sv.drain(60000)
        for r in sv.poll(4096):
            got[r["tag"]] = r

    for rnd in range(4):
        print("ring", rnd, flush=True)
        for k in range(150):  # one at a time: nothing else in flight
            query() if k % 70 != 69 else update()
            settle()
        launches = sv.stats()["launches"]
        for k in range(60):  # arrivals that grid mode cannot keep up with
            query() if k != 50 else update()
        settle()
        assert sv.stats()["launches"] > launches
    st = sv.stats()
    assert st["grid_queries"] > 4 * 140 and st["direct_updates"] >= 4
    sv.close()
    dist = {}
    assert len(got) == len(plan)
    for k, (v, s, t) in plan.items():
        assert got[k]["status"] == 0 and got[k]["version"] == v, (k, got[k])
        if s is None:
            continue
        if (v, s) not in dist:
            dist[v, s] = pyoracle.dijkstra(*versions[v], s)[0]
        assert got[k]["cost"] == (int(dist[v, s][t]) if dist[v, s][t] >= 0 else ddp_amd.INF_COST), (k, v)
    dg.close()
