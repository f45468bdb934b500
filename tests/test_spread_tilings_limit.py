"""Which spreading tilings the libraries of both B-spline orders offer (host only).

An owned core needs at least 8 points per axis and LDS for its points in FP64
beside 64 atoms' spline weights (3 axes, 4 values per point of the order's
stencil, one word of padding) and 21 source words each, 65,792 bytes in all: 2,208
points at order 6 and 2,976 at order 5.  A window of T + 8 points per axis (at
most the grid) needs 64 KiB with the weights, sources and origins of 32 atoms,
and at most three windows over a point.
"""
import ctypes
import itertools
import os

import pytest

from mpidopenmmplugin_amd import _capi

AXES = (6, 12, 16, 20, 24, 30, 36, 40, 48, 50, 54, 60, 64, 72, 80, 90, 96, 100, 108, 120, 128, 144, 160, 180, 192, 240,
        256)


def expected(grid, order):
    out = []
    for m in range(10, 0, -1):
        if any(n % 2 ** m or n // 2 ** m < 6 for n in grid):
            continue
        T = [n // 2 ** m for n in grid]
        points = T[0] * T[1] * T[2]
        if min(T) >= 8 and 8 * (points + 64 * (3 * order * 4 + 1 + 21)) <= 65792:
            assert points <= {6: 2208, 5: 2976}[order]
            out.append((m, 1))
        W = [min(t + 8, n) for t, n in zip(T, grid)]
        if all((w - 1) // t + 1 <= 3 for w, t in zip(W, T)) and \
                8 * (W[0] * W[1] * W[2] + 32 * (3 * order * 4 + 20)) + 32 * 3 * 4 <= 65536:
            out.append((m, 2))
    return out + [(-1, 0)]


@pytest.mark.parametrize("order,name", [(6, "libmpid_hip.so"), (5, "libmpid_hip_order5.so")])
def test_tilings_on_offer(order, name):
    lib = ctypes.CDLL(os.path.join(os.path.dirname(_capi.LIB_PATH), name))
    assert lib.mpid_get_pme_bspline_order() == order
    levels, modes = (ctypes.c_int * 32)(), (ctypes.c_int * 32)()
    largest = 0
    for grid in itertools.product(AXES, AXES[::3], AXES[1::4]):
        count = lib.mpid_spread_tilings((ctypes.c_int * 3)(*grid), 32, levels, modes)
        assert [(levels[i], modes[i]) for i in range(count)] == expected(grid, order), grid
        largest = max([largest] + [grid[0] * grid[1] * grid[2] >> 3 * levels[i] for i in range(count) if modes[i] == 1])
    assert largest > {6: 2100, 5: 2800}[order]  # the grids reach the limit
