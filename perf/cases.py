"""The work that users of this framework have it do, as measurable cases.

Five kinds of calls, each through the package's public entry points:

bfs    hop-count heuristic of one target (DeviceGraph.bfs_hops), whole array back on the host;
astar  one point-to-point query (astar) in an execution mode that suits its graph;
batch  many queries over one resident graph (Batch: upload, launch, wait, download);
dastar one query kept exact over edge updates (DAStar.apply), a batch and its inverse per pass;
serve  a burst of requests with update batches among them (Server.replay).

Graphs are the framework's own generators': random (every node the same
out-degree), maze (4-connected grid with blocked cells and a carved corridor,
unit weights), geometric (points in a square, road-like) and rmat (power law).
A seed gives the graph, the queries and the updates.  Node paths are returned
where weights are spread so widely that shortest paths are unique in practice;
on unit or short integer weights many paths share the least cost, and which of
them comes back is free, so those cases return costs.
"""
import heapq
import math

import numpy as np

import ddp_amd
from ddp_amd import HostGraph

LATTICE = 100000       # the geometric benchmark graph's square
WIDE_LATTICE = 1000000  # with WIDE_UNIT: lengths fine enough for unique paths
WIDE_UNIT = 1000
PATH_CAP = 2048  # longer than any path that is returned
INF = ddp_amd.INF_COST


def listed():
    return [
        # the heuristic array of a single query: the smallest call that touches a whole graph
        {"name": "bfs random 100k", "kind": "bfs", "graph": "random", "n": 100000, "deg": 6, "reverse": True},
        # power-law graph, forward: seven or so very wide levels
        {"name": "bfs rmat 1M", "kind": "bfs", "graph": "rmat", "n": 1 << 20, "deg": 16, "reverse": False},
        # maze: thousands of narrow levels, one after another
        {"name": "bfs maze 2048", "kind": "bfs", "graph": "maze", "n": 2048 * 2048, "deg": 4, "reverse": True},
        # an interactive path request on a small map: latency alone
        {"name": "astar maze 64", "kind": "astar", "graph": "maze", "n": 64 * 64, "deg": 4, "mode": "bidi", "K": 256},
        # the classic GA* query: K lane queues over the GPU, hop-count heuristic
        {"name": "astar random 100k", "kind": "astar", "graph": "random", "n": 100000, "deg": 6, "mode": "grid",
         "K": 1024},
        # corner to corner of the largest maze: a serial chain of thousands of rounds
        {"name": "astar maze 4096", "kind": "astar", "graph": "maze", "n": 4096 * 4096, "deg": 4, "mode": "bidi",
         "K": 512},
        # one full-width query on a power-law graph (a service at low load)
        {"name": "astar rmat 1M", "kind": "astar", "graph": "rmat", "n": 1 << 20, "deg": 16, "mode": "grid",
         "K": 16384},
        # a small batch on a town-sized map, with the paths
        {"name": "batch geo 20k x 64", "kind": "batch", "graph": "geo", "n": 20000, "deg": 10, "queries": 64},
        # the framework's headline: 4,096 queries of all lengths on a country-sized map
        {"name": "batch geo 2M x 4096", "kind": "batch", "graph": "geo", "n": 2000000, "deg": 10, "queries": 4096},
        # all-purpose Dijkstra batch on a power-law graph, h = 0
        {"name": "batch rmat 1M x 256", "kind": "batch", "graph": "rmat", "n": 1 << 20, "deg": 16, "queries": 256},
        # a standing query under 20,000 edge updates at a time
        {"name": "dastar 1M x 20000", "kind": "dastar", "n": 1000000, "deg": 8, "lines": 20000, "mode": "piles",
         "recompute": False},
        # a burst of requests at the server, an update batch among every twenty
        {"name": "serve geo 200k x 1024", "kind": "serve", "graph": "geo", "n": 200000, "deg": 10, "requests": 1024,
         "lines": 200},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["bfs", "astar", "astar", "batch", "batch", "dastar", "serve"])
    if kind == "dastar":
        return {"kind": kind, "n": _log(rng, 2000, 400000), "deg": rng.randint(3, 10), "lines": 2 * _log(rng, 1, 5000),
                "mode": rng.choice(["piles", "grid"]), "recompute": rng.random() < 0.25}
    if kind == "serve":
        return {"kind": kind, "graph": "geo", "n": _log(rng, 5000, 200000), "deg": rng.randint(8, 12),
                "requests": _log(rng, 40, 1000), "lines": 2 * _log(rng, 1, 100)}
    if kind == "batch":
        if rng.random() < 0.3:
            return {"kind": kind, "graph": "rmat", "n": 1 << rng.randint(12, 18), "deg": rng.randint(8, 16),
                    "queries": _log(rng, 8, 256)}
        return {"kind": kind, "graph": "geo", "n": _log(rng, 2000, 1000000), "deg": rng.randint(8, 14),
                "queries": _log(rng, 1, 3000)}
    if kind == "bfs":
        graph = rng.choice(["random", "rmat", "maze", "geo"])
        n = {"random": _log(rng, 500, 1000000), "rmat": 1 << rng.randint(10, 19), "geo": _log(rng, 2000, 500000),
             "maze": _log(rng, 24, 1500) ** 2}[graph]
        deg = {"random": rng.randint(3, 12), "rmat": rng.randint(6, 16), "geo": rng.randint(8, 14), "maze": 4}[graph]
        return {"kind": kind, "graph": graph, "n": n, "deg": deg, "reverse": rng.random() < 0.5}
    graph = rng.choice(["random", "rmat", "maze", "geo"])
    if graph == "maze":
        mode = rng.choice(["bidi", "piles"])
        return {"kind": kind, "graph": graph, "n": _log(rng, 24, 2000) ** 2, "deg": 4, "mode": mode,
                "K": rng.choice([256, 512, 1024])}
    if graph == "geo":
        return {"kind": kind, "graph": graph, "n": _log(rng, 2000, 500000), "deg": rng.randint(8, 14),
                "mode": "piles", "K": 1024}
    if graph == "rmat":
        return {"kind": kind, "graph": graph, "n": 1 << rng.randint(12, 19), "deg": rng.randint(8, 16), "mode": "grid",
                "K": 1 << rng.randint(10, 15)}
    return {"kind": kind, "graph": graph, "n": _log(rng, 1000, 500000), "deg": rng.randint(3, 10),
            "mode": rng.choice(["grid", "piles"]), "K": rng.choice([256, 512, 1000])}


# ------------------------------------------------------------------- inputs

def _unique_paths(case):
    """Whether the case's weights make shortest paths unique in practice."""
    return case.get("graph", "random") == "random" or (case.get("graph") == "geo" and case["n"] <= 50000)


def _graph(case, seed):
    n, deg, kind = case["n"], case["deg"], case.get("graph", "random")
    if kind == "random":
        return HostGraph.random(n, deg, 1000, 100000, seed)
    if kind == "maze":
        side = math.isqrt(n)
        return HostGraph.grid_maze(side, side, 300, seed)
    if kind == "rmat":
        return HostGraph.rmat(n.bit_length() - 1, n * deg, 0.57, 0.19, 0.19, 1, 1000, seed)
    if not _unique_paths(case):
        return HostGraph.geometric(n, deg, LATTICE, seed)
    # travel times: length in thousandths of a lattice unit plus a random delay
    g = HostGraph.geometric(n, deg, WIDE_LATTICE, seed)
    delay = np.random.default_rng(seed).integers(0, WIDE_UNIT, g.E)
    return HostGraph(g.off, g.col, g.w.astype(np.int64) * WIDE_UNIT + delay, xy=g.xy)


def _lattice(case):
    return (WIDE_LATTICE, WIDE_UNIT) if _unique_paths(case) else (LATTICE, 1)


def _pairs(case, hg, nq, seed):
    """Queries as they come: connected, on a map of every length."""
    kind = case.get("graph", "random")
    if kind == "rmat":
        return hg.hub_pairs(nq, seed)
    if kind == "geo":
        side = _lattice(case)[0]
        return hg.geo_pairs(nq, max(side / 1000, 2 * side / math.sqrt(hg.N)), side, seed)
    return hg.reachable_pairs(nq, seed)


def _stroll(hg, off, v, steps, rng):
    """Where a random walk from v ends: a node connected to v."""
    for r in rng.integers(0, 12, steps).tolist():
        if off[v + 1] > off[v]:
            v = int(hg.col[off[v] + r % (off[v + 1] - off[v])])
    return v


def _one_pair(case, hg, seed):
    if case.get("graph") == "maze":  # from about one corner to about the other
        rng, off = np.random.default_rng(seed), hg.offsets_full()
        return tuple(_stroll(hg, off, v, math.isqrt(hg.N), rng) for v in (0, hg.N - 1))
    if case.get("graph") == "geo":  # across a good part of the map
        side = _lattice(case)[0]
        src, dst = hg.geo_pairs(1, side / 2, side, seed)
    else:
        src, dst = _pairs(case, hg, 1, seed)
    return int(src[0]), int(dst[0])


def _bfs_target(case, hg, seed):
    """A node with edges: on a maze, the corridor's start."""
    some = np.flatnonzero(np.diff(hg.offsets_full()))
    return 0 if case["graph"] == "maze" else int(some[np.random.default_rng(seed).integers(0, len(some))])


def _updates(hg, pairs, lines, seed, weight):
    """`pairs` update batches of `lines` lines, half deletes of existing edges
    and half inserts, and for each the batch that undoes it."""
    rng = np.random.default_rng(seed)
    off = hg.offsets_full().astype(np.int64)
    out = []
    half = max(1, lines // 2)
    for _ in range(pairs):
        e = np.unique(rng.integers(0, hg.E, half))
        u = np.searchsorted(off, e, side="right") - 1
        v, w = hg.col[e], hg.w[e]
        # a delete takes the first of parallel edges: keep the edges that are the first
        first = np.array([not np.any(hg.col[off[a]:j] == c) for a, j, c in zip(u, e, v)], bool)
        u, v, w = u[first], v[first], w[first]
        iu = rng.integers(0, hg.N, half)
        iv = rng.integers(0, hg.N, half)
        iw = weight(rng, iu, iv)
        ins = list(zip([1] * half, iu.tolist(), iv.tolist(), iw.tolist()))
        dels = list(zip([0] * len(u), u.tolist(), v.tolist(), [0] * len(u)))
        back = [(0, a, b, 0) for _, a, b, _ in ins] + list(zip([1] * len(u), u.tolist(), v.tolist(), w.tolist()))
        out.append((dels + ins, back))
    return out


def _dastar_inputs(case, seed):
    hg = _graph(case, seed)
    src, dst = hg.reachable_pairs(1, seed)
    ups = _updates(hg, 16, case["lines"], seed + 1, lambda rng, u, v: rng.integers(1000, 100001, len(u)))
    return hg, int(src[0]), int(dst[0]), ups


def _serve_inputs(case, seed):
    hg = _graph(case, seed)
    side, unit = _lattice(case)
    xy = hg.xy.reshape(-1, 2).astype(np.float64)

    def weight(rng, u, v):  # no shorter than the straight line: the heuristic stays a lower bound
        d = np.hypot(*(xy[u] - xy[v]).T)
        return (np.ceil(d).astype(np.int64) + 1) * unit + rng.integers(0, 1000, len(u))

    nreq = case["requests"]
    src, dst = _pairs(case, hg, nreq, seed)
    flat = [b for pair in _updates(hg, max(1, nreq // 40), case["lines"], seed + 1, weight) for b in pair]
    types = np.zeros(nreq, np.int32)
    types[(np.arange(len(flat)) + 1) * nreq // (len(flat) + 1)] = 1
    it = iter(flat)
    return hg, types, src, dst, [next(it) if ty else None for ty in types]


MODES = {"grid": ddp_amd.MODE_GRID, "piles": ddp_amd.MODE_PILES, "bidi": ddp_amd.MODE_BIDI}


def prepare(case, seed):
    kind = case["kind"]
    ctx = ddp_amd.Context(0)
    st = {"case": case, "ctx": ctx}
    if kind == "bfs":
        hg = _graph(case, seed)
        st.update(dg=ddp_amd.DeviceGraph(ctx, hg, reverse=case["reverse"]), t=_bfs_target(case, hg, seed))
        return st
    if kind == "dastar":
        hg, s, t, ups = _dastar_inputs(case, seed)
        # a heuristic that no version of the graph violates: hops over old and new edges together
        off = hg.offsets_full()
        new = np.array([l for pair in ups for l in pair[0] if l[0] == 1], np.int64).reshape(-1, 4)
        us = np.concatenate([np.repeat(np.arange(hg.N), np.diff(off)), new[:, 1]])
        order = np.argsort(us, kind="stable")
        union = HostGraph(np.searchsorted(us[order], np.arange(hg.N)).astype(np.int32),
                          np.concatenate([hg.col, new[:, 2].astype(np.int32)])[order],
                          np.concatenate([hg.w, new[:, 3].astype(np.uint32)])[order])
        ug = ddp_amd.DeviceGraph(ctx, union, reverse=True)
        h, _ = ug.bfs_hops(t, reverse=True, scale=1000)
        ug.close()
        mode = MODES[case["mode"]]
        st.update(d=ddp_amd.DAStar(ctx, hg, s, t, h=h, K=1024 if case["n"] < 100000 else 16384, mode=mode),
                  ups=ups, at=0, how=ddp_amd.DAStar.RECOMPUTE if case["recompute"] else ddp_amd.DAStar.REPAIR)
        return st
    if kind == "serve":
        hg, types, src, dst, ups = _serve_inputs(case, seed)
        dg = ddp_amd.DeviceGraph(ctx, hg, reorder=True)
        sv = ddp_amd.Server(ctx, dg, heur=ddp_amd.H_EUCLID, scale=_lattice(case)[1], idle_ms=2)
        st.update(dg=dg, sv=sv, types=types, src=src, dst=dst, ups=ups, arrival=np.zeros(len(types)))
        return st
    hg = _graph(case, seed)
    graph = case["graph"]
    if kind == "batch":
        src, dst = _pairs(case, hg, case["queries"], seed)
        dg = ddp_amd.DeviceGraph(ctx, hg, reorder=True)
        heur = ddp_amd.H_EUCLID if graph == "geo" else ddp_amd.H_ZERO
        cap = PATH_CAP if _unique_paths(case) else 0
        b = ddp_amd.Batch(ctx, dg, len(src), heur=heur, scale=_lattice(case)[1] if graph == "geo" else 1, path_cap=cap)
        st.update(dg=dg, b=b, src=src, dst=dst, cap=cap)
        return st
    s, t = _one_pair(case, hg, seed)
    K, scale, heap_cap = case["K"], 1, 0
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=graph in ("maze", "random"), reorder=graph in ("geo", "rmat"))
    if graph == "maze":
        dg.set_grid(math.isqrt(case["n"]))
        heur = ddp_amd.H_MANHATTAN
    elif graph == "geo":
        heur, scale = ddp_amd.H_EUCLID, _lattice(case)[1]
    elif graph == "random":
        dg.bfs_hops(t, reverse=True, scale=1000, store_as_h=True, want=False)
        heur = ddp_amd.H_ARRAY
    else:
        heur = ddp_amd.H_ZERO
        heap_cap = max(2 * hg.N // K + 256, (8 * hg.N + K - 1) // K)  # hubs are queued many times
    st.update(dg=dg, args=dict(s=s, t=t, heur=heur, scale=scale, K=K, heap_cap=heap_cap, mode=MODES[case["mode"]],
                               path_cap=None if _unique_paths(case) else 0))
    return st


# --------------------------------------------------------------------- pass

def _row(path, cap):
    """A node path in a row of cap entries, -1 behind it."""
    return np.pad(path, (0, cap - len(path)), constant_values=-1)


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "bfs":
        hops, levels = st["dg"].bfs_hops(st["t"], reverse=case["reverse"])
        return {"hops": hops, "levels": levels}
    if kind == "astar":
        r = ddp_amd.astar(st["ctx"], st["dg"], **st["args"])
        return {"cost": r.cost, "path": _row(r.path, PATH_CAP)} if _unique_paths(case) else {"cost": r.cost}
    if kind == "batch":
        b = st["b"]
        b.upload(st["src"], st["dst"])
        b.launch()
        b.wait()
        out = b.download(paths=st["cap"] > 0)
        res = {"cost": out["cost"], "error": out["qerr"]}
        if st["cap"]:
            res["paths"] = np.stack([_row(p, st["cap"]) for p in out["paths"]])
        return res
    if kind == "dastar":
        there, back = st["ups"][st["at"] % len(st["ups"])]
        st["at"] += 1
        c1, s1 = st["d"].apply(there, mode=st["how"])
        path = st["d"].path()
        c2, s2 = st["d"].apply(back, mode=st["how"])
        return {"cost": [c1, c2], "path": _row(path, PATH_CAP), "deleted": [s1["deletes_effective"], s2["deletes_effective"]]}
    res = st["sv"].replay(st["arrival"], st["types"], st["src"], st["dst"], st["ups"])
    return {"cost": np.array([r["cost"] for r in res], np.int32),
            "status": np.array([r["status"] for r in res], np.int32)}


def work(case):
    """Each row of the graph read once, each answer written once."""
    n = case["n"]
    e = n * case["deg"] * (0.49 if case.get("graph") == "maze" else 1)
    kind = case["kind"]
    if kind == "bfs":
        return {"bytes": 8 * n + 4 * e, "flops": 0}
    if kind == "dastar":
        # the lines, both rows of each line's nodes and their words
        return {"bytes": 2 * case["lines"] * (16 + 2 * 8 * case["deg"] + 16), "flops": 0}
    rows = 4 * n + 8 * e + (8 * n if case["graph"] == "geo" else 0) + (4 * n if case["graph"] == "random" else 0)
    answers = 4 * case.get("queries", 1) + 4 * case.get("requests", 0)
    return {"bytes": rows + answers, "flops": 0}


# ------------------------------------------------------------------- exact

def _hops(off, col, t):
    dist = np.full(len(off) - 1, -1, np.int64)
    dist[t] = 0
    front, level = np.array([t]), 0
    while len(front):
        level += 1
        lens = off[front + 1] - off[front]
        at = np.repeat(off[front] - np.concatenate([[0], np.cumsum(lens)[:-1]]), lens) + np.arange(lens.sum())
        nxt = np.unique(col[at])
        front = nxt[dist[nxt] < 0]
        dist[front] = level
    return dist, level


def _dijkstra(off, col, w, s, t):
    dist, heap = {s: 0}, [(0, s)]
    while heap:
        d, u = heapq.heappop(heap)
        if u == t:
            return d
        if d > dist[u]:
            continue
        for j in range(off[u], off[u + 1]):
            v, x = col[j], d + w[j]
            if x < dist.get(v, INF):
                dist[v] = x
                heapq.heappush(heap, (x, v))
    return INF


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("bfs", "astar", "batch") or case["n"] > (200000 if kind == "astar" else 1100000):
        return None
    if kind == "batch" and case["n"] * case["queries"] > 1500000:
        return None
    hg = _graph(case, seed)
    off = hg.offsets_full().astype(np.int64)
    if kind == "bfs":
        col = hg.col.astype(np.int64)
        if case["graph"] == "maze" and hg.N > 250000:
            return None
        if case["reverse"]:
            order = np.argsort(col, kind="stable")
            back = np.repeat(np.arange(hg.N), np.diff(off))[order]
            off, col = np.searchsorted(col[order], np.arange(hg.N + 1)), back
        hops, levels = _hops(off, col, _bfs_target(case, hg, seed))
        return {"hops": hops, "levels": levels}
    off, col, w = off.tolist(), hg.col.tolist(), hg.w.tolist()
    if kind == "astar":
        return {"cost": _dijkstra(off, col, w, *_one_pair(case, hg, seed)), "path": None}
    src, dst = _pairs(case, hg, case["queries"], seed)
    return {"cost": np.array([_dijkstra(off, col, w, int(a), int(b)) for a, b in zip(src, dst)], np.int64),
            "error": None}
