"""Row location and edge collection of the slot engines at the sizes
where they can go wrong: rows of 0, 1, 63, 64, 65, 127, 128 and hundreds of
edges side by side, rounds from one row to more edges than a wave collects,
deleted edges, and the relaxation by compare-and-swap (zero weights).  Costs
are exact integers and equal the oracle's."""
import numpy as np
import pytest

import ddp_amd
from helpers import path_cost
from oracle import pyoracle

pytestmark = pytest.mark.gpu

PATTERNS = {
    "ones": [1, 1, 1, 1],
    "empty": [0, 0, 3, 0, 1, 0],
    "sixtyfour": [64, 64, 128, 64],
    "around": [63, 65, 1, 64, 127, 0, 128, 2],
    "hubs": [700, 1, 0, 2, 1500, 5],
}


def graph(rng, N, lens, wmin):
    deg = np.asarray([lens[i % len(lens)] for i in range(N)])
    deg[0] = min(N, 200)  # a first round of some width
    off = np.zeros(N, np.int32)
    off[1:] = np.cumsum(deg)[:-1]
    col = rng.integers(0, N, int(deg.sum())).astype(np.int32)
    # non-empty rows also lead on, so that searches go deep
    for u in np.flatnonzero(deg):
        col[off[u]] = (u + 1 + rng.integers(0, 3)) % N
    col[rng.random(len(col)) < 0.03] = -1
    return off, col, rng.integers(wmin, 60, len(col)).astype(np.uint32)


@pytest.mark.parametrize("block", [64, 256, 512, 1024])
@pytest.mark.parametrize("lens", list(PATTERNS))
@pytest.mark.parametrize("wmin", [0, 1])
def test_rows_of_all_lengths(ctx, block, lens, wmin):
    rng = np.random.default_rng(len(lens) * 7 + block + wmin)
    hg = ddp_amd.HostGraph(*graph(rng, 1200, PATTERNS[lens], wmin))
    dg = ddp_amd.DeviceGraph(ctx, hg)
    src = np.concatenate([np.zeros(8), rng.integers(0, hg.N, 16)]).astype(np.int32)
    dst = rng.integers(0, hg.N, 24).astype(np.int32)
    want = []
    for s, t in zip(src, dst):
        d, _ = pyoracle.dijkstra(hg.off, hg.col, hg.w, int(s), int(t))
        want.append(int(d[t]) if d[t] >= 0 else ddp_amd.INF_COST)
    for engine in (ddp_amd.ENGINE_PILES, ddp_amd.ENGINE_HEAPS):
        print("rows", block, lens, wmin, engine, flush=True)
        costs, paths, st = ddp_amd.astar_batch(ctx, dg, src, dst, heur=ddp_amd.H_ZERO, block=block, slots=6,
                                               path_cap=hg.N + 1, engine=engine)
        assert st["errors"] == 0
        assert np.array_equal(costs, np.asarray(want))
        for i, p in enumerate(paths):
            if want[i] != ddp_amd.INF_COST:
                assert p[0] == src[i] and p[-1] == dst[i]
                assert path_cost(hg.off, hg.col, hg.w, p) == want[i]
    dg.close()


@pytest.mark.parametrize("block", [256, 512, 1024])
@pytest.mark.parametrize("lens", list(PATTERNS))
@pytest.mark.parametrize("wmin", [0, 1])
def test_rows_of_all_lengths_bidi(ctx, block, lens, wmin):
    rng = np.random.default_rng(len(lens) * 11 + block + wmin)
    hg = ddp_amd.HostGraph(*graph(rng, 1200, PATTERNS[lens], wmin))
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=True)
    src = np.concatenate([np.zeros(8), rng.integers(0, hg.N, 16)]).astype(np.int32)
    dst = rng.integers(0, hg.N, 24).astype(np.int32)
    print("rows bidi", block, lens, wmin, flush=True)
    costs, paths, st = ddp_amd.astar_batch(ctx, dg, src, dst, heur=ddp_amd.H_ZERO, block=block, slots=6,
                                           path_cap=2 * hg.N + 1, engine=ddp_amd.ENGINE_BIDI)
    assert st["errors"] == 0
    for i, (s, t) in enumerate(zip(src, dst)):
        d, _ = pyoracle.dijkstra(hg.off, hg.col, hg.w, int(s), int(t))
        want = int(d[t]) if d[t] >= 0 else ddp_amd.INF_COST
        assert costs[i] == want
        if want != ddp_amd.INF_COST:
            assert paths[i][0] == s and paths[i][-1] == t
            assert path_cost(hg.off, hg.col, hg.w, paths[i]) == want
    dg.close()
