"""Level-synchronous BFS at the sizes where its paths change: rows around the
length at which they are cut into segments, levels around the widths at which
the narrow grid hands over to the wide one and back, and the allocation-free
variant's longer segments.  Checked against the oracle's BFS."""
import ctypes
from ctypes import byref, c_int32, c_void_p

import numpy as np
import pytest

import ddp_amd
from ddp_amd import _capi
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def star(deg, n, deleted=0):
    """Node 0 points at deg nodes (i % n), the first `deleted` of the edges deleted; node 1 back at 0."""
    col = (np.arange(deg, dtype=np.int64) % n).astype(np.int32)
    col[:deleted] = -1
    off = np.full(n, deg, np.int32)
    off[0] = 0
    off[2:] = deg + 1
    return ddp_amd.HostGraph(off, np.append(col, 0), np.ones(deg + 1))


def layers(width, depth):
    """Node 0 to `width` nodes, each of them to one node of the next layer, the last layer to one sink."""
    n = 2 + width * depth
    rows = [1 + np.arange(width)]
    for k in range(depth - 1):
        rows.append(1 + (k + 1) * width + np.arange(width))
    rows.append(np.full(width, n - 1))
    off = np.zeros(n, np.int32)
    off[1:n - 1] = width + np.arange(width * depth)
    off[n - 1] = width * (depth + 1)
    return ddp_amd.HostGraph(off, np.concatenate(rows), np.ones(width * (depth + 1)))


@pytest.mark.parametrize("hg,t", [
    (star(63, 70), 0), (star(64, 70), 1), (star(65, 70), 1), (star(129, 1000, deleted=66), 1),
    (star(4096 * 64, 300000), 0), (star(4096 * 64 + 1, 300000), 1), (star(1000000, 5000), 1),
    (layers(2047, 3), 0), (layers(2048, 3), 0), (layers(2049, 3), 0), (layers(4096, 2), 0), (layers(4097, 4), 0),
    (layers(70000, 2), 0), (layers(1, 40), 0),
], ids=lambda x: f"N{x.N}-E{x.E}" if isinstance(x, ddp_amd.HostGraph) else str(x))
def test_bfs_segments_and_grids(ctx, hg, t):
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=True)
    for reverse, gg in ((False, hg), (True, hg.transpose())):
        want, levels = pyoracle.bfs_hops(gg.off, gg.col, t)
        got, lv = dg.bfs_hops(t, reverse=reverse)
        assert lv == levels and np.array_equal(got, want)
    dg.close()


def test_bfs_noalloc_long_rows(ctx):
    hip = ctypes.CDLL("libamdhip64.so")
    hg = star(17000000, 100000)  # more than the scratch holds in segments of the default length
    dg = ddp_amd.DeviceGraph(ctx, hg)
    want, levels = dg.bfs_hops(1)
    buf, lv = c_void_p(), c_int32()
    assert hip.hipMalloc(byref(buf), ctypes.c_size_t(4 * hg.N)) == 0
    got = np.empty(hg.N, np.int32)
    try:
        assert _capi.lib().ddp_bfs_hops_noalloc(ctx.handle, dg.handle, 1, 0, 1, buf, byref(lv)) == 0
        assert hip.hipMemcpy(got.ctypes.data_as(c_void_p), buf, ctypes.c_size_t(4 * hg.N), 2) == 0
    finally:
        hip.hipFree(buf)
    assert lv.value == levels == 3 and np.array_equal(got, want)
    assert got[1] == 0 and got[0] == 1 and (got[2:] == 2).all()
    dg.close()
