"""Strips of a level that does not fit the chip (host side): the strips cover the
level, each region holds its strip's rows and as many beyond them as a round
has sweeps, the exchange planes fit the scratch, and the rounds add up."""
import ctypes

import pytest


@pytest.mark.parametrize("fma", [0, 1])
def test_strips_cover_with_their_cuts(vsc, fma):
    L = vsc.lib()
    out, xs, ys = (ctypes.c_int * 8)(), (ctypes.c_int * 1024)(), (ctypes.c_int * 1024)()
    found = 0
    for W in (1281, 1920, 2001, 2560, 3000, 3840, 5120, 7680):
        for H in (720, 1001, 1125, 1440, 2160, 2250, 4320):
            for iters in (1, 20, 31, 75, 100, 149, 150, 300):
                if not L.vsct_resident_strips(W, H, iters, 256, fma, out, xs, ys):
                    continue
                found += 1
                tw, th, h, nx, ny, rounds, strips, rows = out
                sweeps = -(-iters // rounds)
                own = -(-H // strips)
                assert rows <= H and 3 * nx * ny <= 256 and (rounds - 1) * sweeps < iters
                assert (1 if fma and rounds == 1 else 2 if fma else 4) * rows <= H
                assert list(xs[:nx])[-1] == W - tw and list(ys[:ny])[-1] == rows - th
                for k in range(strips):
                    y0, y1 = min(k * own, H), min((k + 1) * own, H)
                    top = max(0, min(y0 - sweeps, H - rows))
                    assert top + rows <= H
                    if y0 < y1:
                        assert top == 0 or top <= y0 - sweeps
                        assert top + rows == H or top + rows >= y1 + sweeps
    assert found > (10 if fma else 0)
    # levels that are faster blocked, too small for strips, or have no sweeps
    assert not L.vsct_resident_strips(640, 360, 150, 256, fma, out, xs, ys)
    assert not L.vsct_resident_strips(3840, 2160, 0, 256, fma, out, xs, ys)
