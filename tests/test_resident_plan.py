"""Tilings of the resident consistency solver (host side): every tile lies in
the level, the tiles' exact parts cover it, and every pixel of a tile's halo is
in the exact part of the neighbour that publishes it, for all the sizes and
sweep counts a frame can ask for."""
import ctypes

import pytest


def _plan(vsc, W, H, iters, cus, fma):
    L = vsc.lib()
    out, xs, ys = (ctypes.c_int * 5)(), (ctypes.c_int * 1024)(), (ctypes.c_int * 1024)()
    if not L.vsct_resident_plan(W, H, iters, cus, fma, out, xs, ys):
        return None
    tw, th, h, nx, ny = out
    return tw, th, h, list(xs[:nx]), list(ys[:ny])


def _axis(L, T, h, starts):
    n = len(starts)
    exact = [(s + (0 if i == 0 else h), s + T - (0 if i == n - 1 else h)) for i, s in enumerate(starts)]
    assert starts[0] == 0 and starts[-1] == L - T
    at = 0
    for i, s in enumerate(starts):
        assert 0 <= s <= L - T
        assert exact[i][0] <= at or i == 0
        at = max(at, exact[i][1])
        if i > 0:       # the halo towards the tile before lies in that tile's exact part
            assert exact[i - 1][0] <= s and s + h <= exact[i - 1][1]
        if i < n - 1:
            assert exact[i + 1][0] <= s + T - h and s + T <= exact[i + 1][1]
    assert at == L


@pytest.mark.parametrize("fma", [0, 1])
@pytest.mark.parametrize("cus", [256, 64, 32])
def test_tilings_cover_and_exchange(vsc, fma, cus):
    sizes = [(W, H) for W in (64, 65, 99, 127, 128, 129, 131, 255, 256, 257, 300, 480, 640, 853, 960, 1281, 1571, 1920)
             for H in (32, 33, 45, 47, 48, 49, 63, 64, 101, 129, 180, 270, 361, 540, 719, 784, 1080)]
    found = 0
    for W, H in sizes:
        for iters in (1, 2, 7, 20, 75, 149, 150, 304):
            p = _plan(vsc, W, H, iters, cus, fma)
            if p is None:
                continue
            found += 1
            tw, th, h, xs, ys = p
            assert h % 4 == 0 and 3 * len(xs) * len(ys) <= min(cus, 1024)
            assert tw >= 4 * h and th >= 4 * h
            for s in xs[:-1]:
                assert s % 4 == 0     # a lane's pixels are wholly exact or wholly halo
            _axis(W, tw, h, xs)
            _axis(H, th, h, ys)
    assert found > 100
    # a level narrower or lower than every tile, or one that does not fit the chip, has none
    assert _plan(vsc, 63, 500, 150, cus, fma) is None and _plan(vsc, 500, 31, 150, cus, fma) is None
    assert _plan(vsc, 3840, 2160, 150, cus, fma) is None and _plan(vsc, 640, 360, 0, cus, fma) is None
