"""Update lines from Python objects to the ABI's structs: the native conversion
gives what one ctypes store per field gives, for every kind of line."""
import ctypes
import struct

import numpy as np
import pytest

import ddp_amd
from ddp_amd import _capi


def by_field(lines):
    arr = (_capi.Update * max(1, len(lines)))()
    for i, l in enumerate(lines):
        arr[i].flag, arr[i].u, arr[i].v, arr[i].w = int(l[0]), int(l[1]), int(l[2]), int(l[3])
    return bytes(arr)


@pytest.mark.parametrize("lines", [
    [], [(1, 2, 3, 4)], [[0, 5, 6, 0], (1, 7, 8, 2 ** 32 - 1)], ((1, 2 ** 31 - 1, -1, 5), (0, -2 ** 31, 0, -3)),
    [(1, 2, 3, 2 ** 40 + 7)], [(1, 2, 3, 2 ** 70 + 9)], [(1, 2, 3, 4, 5)], [(True, 2, 3, 4)], [(1, 2.9, 3, 4)],
    [(np.int32(1), np.int64(2), np.uint8(3), 4)], np.arange(40).reshape(10, 4), [("1", "2", "3", "4")],
    [tuple(int(x) for x in r) for r in np.random.default_rng(1).integers(-2 ** 33, 2 ** 33, (3000, 4))],
], ids=lambda v: f"{type(v).__name__}{len(v)}")
def test_updates_array(lines):
    assert bytes(ddp_amd._updates_array(lines)) == by_field(lines)


@pytest.mark.parametrize("lines,error", [([(1, 2, 3)], IndexError), ([(1, 2, 3, None)], TypeError),
                                         ([(1, 2, 3, "x")], ValueError), ([5], TypeError), (None, TypeError)])
def test_updates_array_refuses(lines, error):
    with pytest.raises(error):
        ddp_amd._updates_array(lines)


def test_result_dicts():
    assert struct.calcsize(_capi.SERVER_RESULT_FORMAT) == ctypes.sizeof(_capi.ServerResult)
    arr = (_capi.ServerResult * 3)()
    for i, r in enumerate(arr):
        r.tag, r.type, r.cost, r.version, r.status = 2 ** 63 + i, i, -i, 7, 16
        r.submit_ms, r.done_ms, r.device_ms = 0.25 * i, 1.5, -2.0
    got = ddp_amd._result_dicts(arr, 2)
    assert got == [{f: getattr(r, f) for f, _ in _capi.ServerResult._fields_} for r in arr[:2]]
