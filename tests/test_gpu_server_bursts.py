"""Serving bursts and update batches at the sizes where the claim and update
paths change: more requests than one poll copies (64) or the ring holds,
sources with many inserts in one batch, rows and parallel edges around the
groups of 8 that deletes scan.  Every query against Dijkstra on its version."""
import numpy as np
import pytest

import ddp_amd
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def trace(n, per_source, seed):
    """A graph whose first 32 rows are 0..31 edges long (some parallel), and per
    burst position a query or an update: `per_source` inserts from one node,
    single ones from others, deletes of parallel and of just inserted edges."""
    rng = np.random.default_rng(seed)
    deg = np.concatenate([np.arange(32), rng.integers(1, 6, n - 32)])
    off = np.concatenate([[0], np.cumsum(deg)[:-1]]).astype(np.int32)
    col = rng.integers(0, n, deg.sum()).astype(np.int32)
    for u in range(9, 32, 3):  # the same edge at both ends of the row
        col[off[u] + deg[u] - 1] = col[off[u]]
    hg = ddp_amd.HostGraph(off, col, rng.integers(1, 50, deg.sum()))
    updates = []
    for k in range(6):
        lines = [(1, 7, int(rng.integers(0, n)), int(rng.integers(1, 50))) for _ in range(per_source)]
        lines += [(1, int(u), int(rng.integers(0, n)), int(rng.integers(1, 50))) for u in rng.integers(0, n, 40)]
        for u in (int(x) for x in rng.integers(1, 32, 12)):
            lines += [(0, u, int(hg.col[off[u] + j]), 0) for j in (0, deg[u] - 1)]
        if updates:  # inserted by the batch before
            lines += [(0, l[1], l[2], 0) for l in updates[-1] if l[0] == 1][::3]
        updates.append(lines)
    return hg, updates


@pytest.mark.parametrize("per_source,ring,block,engine", [
    (1, 64, 64, ddp_amd.ENGINE_PILES), (2, 128, 256, ddp_amd.ENGINE_PILES), (65, 1024, 64, ddp_amd.ENGINE_HEAPS),
    (130, 0, 1024, ddp_amd.ENGINE_PILES), (70, 64, 256, ddp_amd.ENGINE_BIDI)])
def test_server_burst(ctx, per_source, ring, block, engine):
    hg, updates = trace(700, per_source, per_source)
    versions = [(hg.off, hg.col, hg.w)]
    for u in updates:
        versions.append(pyoracle.apply_batch(*versions[-1], u)[:3])
    rng = np.random.default_rng(5)
    nreq = 330
    types = np.zeros(nreq, np.int32)
    types[[20, 21, 90, 155, 220, 300]] = 1  # two in a row, and on both sides of 64-entry copies
    src, dst = rng.integers(0, 40, nreq), rng.integers(0, hg.N, nreq)
    it = iter(updates)
    ups = [next(it) if ty else None for ty in types]
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=True)
    sv = ddp_amd.Server(ctx, dg, heur=ddp_amd.H_ZERO, block=block, engine=engine, ring=ring, slots=40, idle_ms=20)
    res = sv.replay(np.zeros(nreq), types, src, dst, ups)
    assert sv.info()["version"] == len(updates)
    sv.close()
    dist, v = {}, 0
    for i, r in enumerate(res):
        v += int(types[i])
        assert r["status"] == 0 and r["version"] == v
        if types[i]:
            continue
        if (v, src[i]) not in dist:
            dist[v, src[i]] = pyoracle.dijkstra(*versions[v], int(src[i]))[0]
        d = dist[v, src[i]][dst[i]]
        assert r["cost"] == (int(d) if d >= 0 else ddp_amd.INF_COST), (i, v)
    dg.close()
