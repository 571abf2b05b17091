"""Tilings of the resident consistency solver (host side): a tile orders its
publications and its last store after its eight neighbours' loads and after no
others', so along an axis the exact part of a tile may not reach the pixels of a
tile two or more away.  Sizes where three tiles overlap by more than that exist
in both solver forms: 64-row tiles on 105 to 115 rows, 48-row ones on 81 to 87."""
import ctypes

import pytest


def _axes(vsc, entry, ints, W, H, iters, cus, fma):
    out, xs, ys = (ctypes.c_int * ints)(), (ctypes.c_int * 1024)(), (ctypes.c_int * 1024)()
    if not entry(W, H, iters, cus, fma, out, xs, ys):
        return []
    tw, th, h, nx, ny = out[:5]
    return [(tw, h, list(xs[:nx])), (th, h, list(ys[:ny]))]


def _apart(T, h, starts):
    n = len(starts)
    for i, a in enumerate(starts):
        exact = (a + (0 if i == 0 else h), a + T - (0 if i == n - 1 else h))
        for j, b in enumerate(starts):
            if abs(i - j) >= 2 and exact[0] < b + T and b < exact[1]:
                return False
    return True


@pytest.mark.parametrize("fma", [0, 1])
@pytest.mark.parametrize("cus", [256, 64])
def test_exact_parts_stay_off_tiles_further_away(vsc, fma, cus):
    L = vsc.lib()
    sizes = [(200, 113), (192, 108), (200, 112), (400, 225), (165, 83), (165, 84), (64, 105), (640, 115)]
    sizes += [(W, H) for W in range(64, 700, 23) for H in range(40, 400, 7)]
    sizes += [(W, H) for W in range(700, 2000, 139) for H in range(300, 1100, 41)]
    found = 0
    for W, H in sizes:
        for iters in (9, 33, 75, 150):
            for T, h, starts in _axes(vsc, L.vsct_resident_plan, 5, W, H, iters, cus, fma):
                found += 1
                assert _apart(T, h, starts), (W, H, iters, T, h, starts)
    assert found > 1000


@pytest.mark.parametrize("fma", [0, 1])
def test_exact_parts_of_strips_stay_off_tiles_further_away(vsc, fma):
    L = vsc.lib()
    found = 0
    for W in range(1100, 7700, 173):
        for H in (720, 1001, 1125, 1301, 1440, 1800, 2160, 2250, 3000, 4320):
            for iters in (20, 31, 50, 75, 150):
                for T, h, starts in _axes(vsc, L.vsct_resident_strips, 8, W, H, iters, 256, fma):
                    found += 1
                    assert _apart(T, h, starts), (W, H, iters, T, h, starts)
    assert found > (100 if fma else 10)
