"""Strips of a level that does not fit the chip (host side).  A strip's region is
swept as an image of its own, whose row 0 has no upper neighbour and whose row
H-2 has no lower one (flowconsistency.cu:215-236), so the values that the cuts
make wrong start a row further in at the bottom.  The rows that a strip keeps
have to be those of the whole level after every sweep of a round."""
import ctypes

import numpy as np
import pytest


def _strips(vsc, W, H, iters, fma):
    L = vsc.lib()
    out, xs, ys = (ctypes.c_int * 8)(), (ctypes.c_int * 1024)(), (ctypes.c_int * 1024)()
    if not L.vsct_resident_strips(W, H, iters, 256, fma, out, xs, ys):
        return None
    rounds, strips, rows = out[5:8]
    sweeps, own = -(-iters // rounds), -(-H // strips)
    regions = []
    for k in range(strips):
        y0, y1 = min(k * own, H), min((k + 1) * own, H)
        if y0 < y1:
            regions.append((max(0, min(y0 - sweeps, H - rows)), y0, y1))
    return sweeps, rows, regions


def _sweep(o, u, q, k, step, mom):
    s = np.zeros_like(o)
    s[1:] += o[:-1]
    s[:-2] += o[1:-1]          # row H-1 is nobody's lower neighbour
    sg = step * (s - q * o) - k
    return o + sg + mom * u, sg


def _bottom_row_rule(o):
    """Rows whose lower neighbour counts: all but the last two."""
    n = len(o)
    return np.arange(n) < n - 2


def test_model_of_a_sweep():
    o = np.arange(1.0, 7.0)
    got, _ = _sweep(o, 0 * o, 0 * o, 0 * o, 1.0, 0.0)
    want = o + np.concatenate([[0], o[:-1]]) + np.where(_bottom_row_rule(o), np.concatenate([o[1:], [0]]), 0)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("fma", [0, 1])
def test_cuts_do_not_reach_the_kept_rows(vsc, fma):
    found = 0
    for W in (1920, 2304, 2563, 3001, 3840, 5120, 7680):
        for H in (720, 1000, 1301, 1439, 2160, 2250, 4320):
            for iters in (12, 16, 20, 31, 50, 101, 149, 150):
                p = _strips(vsc, W, H, iters, fma)
                if p is None:
                    continue
                found += 1
                sweeps, rows, regions = p
                for top, y0, y1 in regions:
                    # first and last row of the region that are right after the round: a cut's rows are wrong
                    # after the first sweep (one above, two below), one more after each
                    lo = top + sweeps if top > 0 else 0
                    hi = top + rows - 1 - sweeps if top + rows < H else H
                    assert lo <= y0 and y1 <= hi, (W, H, iters, sweeps, rows, top, y0, y1)
    assert found > 10


def test_kept_rows_equal_the_whole_level(vsc):
    """A column of the level in 64 bits, with a step that lets a cut be seen after 12 sweeps."""
    H, iters = 2160, 12
    sweeps, rows, regions = _strips(vsc, 3840, H, iters, 1)
    assert sweeps == iters
    rng = np.random.default_rng(5)
    o, q, k = rng.uniform(0, 1, H), rng.uniform(4, 5, H), rng.uniform(-0.1, 0.1, H)

    def level(o, q, k):
        u = np.zeros_like(o)
        for _ in range(iters):
            o, u = _sweep(o, u, q, k, 0.2, 0.15)
        return o

    whole = level(o, q, k)
    for top, y0, y1 in regions:
        part = level(o[top:top + rows], q[top:top + rows], k[top:top + rows])
        assert np.array_equal(part[y0 - top:y1 - top], whole[y0:y1]), (top, y0, y1)
