"""Whole-GPU kernels beside other work on the same GPU: with some of the CUs held
by a serving kernel of another context, and two at once from two contexts.
They run on what is resident (grid_team.h), without waiting for the rest."""
import threading
import time

import numpy as np
import pytest

import ddp_amd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def big():
    """Enough edges for the widest grids (4.2M and more)."""
    hg = ddp_amd.HostGraph.random(600000, 8, 1000, 100000, 5)
    src, dst = hg.reachable_pairs(1, 5)
    return hg, int(src[0]), int(dst[0])


class Calls:
    """The whole-GPU calls of one context, and their answers."""

    def __init__(self, ctx, big):
        self.ctx, (self.hg, self.s, self.t) = ctx, big
        self.dg = ddp_amd.DeviceGraph(ctx, self.hg, reverse=True)
        self.dg.bfs_hops(self.t, reverse=True, scale=1000, store_as_h=True, want=False)
        # opened here: opening and closing free memory, which waits for the whole GPU
        self.d = ddp_amd.DAStar(ctx, self.hg, self.s, self.t, K=16384)

    def bfs(self):
        hops, levels = self.dg.bfs_hops(self.t, reverse=True)
        return int(hops.sum()), levels

    def grid(self, heur):
        return ddp_amd.astar(self.ctx, self.dg, self.s, self.t, heur=heur, K=16384, path_cap=0,
                             mode=ddp_amd.MODE_GRID).cost

    def dastar(self):
        j = 8 * self.s
        v, w = int(self.hg.col[j]), int(self.hg.w[j])
        return [self.d.apply([l], mode=how)[0] for how in (ddp_amd.DAStar.REPAIR, ddp_amd.DAStar.RECOMPUTE)
                for l in ((0, self.s, v, 0), (1, self.s, v, w))]

    def close(self):
        self.d.close()
        self.dg.close()

    def all(self):
        out = []
        for name, f in (("bfs", self.bfs), ("grid h", lambda: self.grid(ddp_amd.H_ARRAY)),
                        ("grid 0", lambda: self.grid(ddp_amd.H_ZERO)), ("dastar", self.dastar)):
            t0 = time.perf_counter()
            out.append((name, f(), time.perf_counter() - t0))
        return out


def test_beside_a_server(ctx, big):
    calls = Calls(ctx, big)
    calls.all()
    alone = calls.all()
    small = ddp_amd.HostGraph.random(2000, 5, 1, 100, 6)
    for slots in (64, 160, 224):
        other = ddp_amd.Context(0)
        sg = ddp_amd.DeviceGraph(other, small)
        sv = ddp_amd.Server(other, sg, heur=ddp_amd.H_ZERO, slots=slots, idle_ms=8000)
        (r,) = sv.replay(np.zeros(1), np.zeros(1, np.int32), [1], [2], [None])  # its slots are up, and wait
        assert r["status"] == 0 and sv.info()["slots"] == slots
        t0 = time.perf_counter()
        shared = calls.all()
        took = time.perf_counter() - t0
        print(slots, [(n, f"{a * 1e3:.2f}", f"{b * 1e3:.2f} ms") for (n, _, a), (_, _, b) in zip(alone, shared)], flush=True)
        (r,) = sv.replay(np.zeros(1), np.zeros(1, np.int32), [1], [2], [None])
        assert r["status"] == 0 and sv.stats()["launches"] == 1  # it was there all the time
        sv.close()
        sg.close()
        other.close()
        assert [(n, x) for n, x, _ in shared] == [(n, x) for n, x, _ in alone]
        assert took < 6  # less than the server's idle time
    calls.close()


def test_two_contexts_at_once(ctx, big):
    calls = Calls(ctx, big)
    want = [(n, x) for n, x, _ in calls.all()]
    got, errors = [], []

    def work():
        try:
            c = ddp_amd.Context(0)
            mine = Calls(c, big)
            for _ in range(4):
                got.append([(n, x) for n, x, _ in mine.all()])
            mine.close()
            c.close()
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=work) for _ in range(2)]
    t0 = time.perf_counter()
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print(f"{time.perf_counter() - t0:.2f} s", flush=True)
    assert not errors, errors
    assert len(got) == 8 and all(g == want for g in got)
    assert time.perf_counter() - t0 < 15
    calls.close()
