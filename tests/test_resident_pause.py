"""Frames that the blocked solver takes after a resident launch that the device
could not hold at once (host side)."""
import ctypes


def _run(vsc, n, given_up):
    a, b = (ctypes.c_ubyte * n)(), (ctypes.c_ubyte * n)()
    for i in given_up:
        a[i] = 1
    vsc.lib().vsct_resident_pause(a, n, b)
    return list(b)


def test_pause_doubles_while_launches_are_given_up(vsc):
    at, expect, i = [], [], 0
    for k in (64, 128, 256, 512, 1024, 2048, 4096, 4096):
        at.append(i)
        expect += [0] * k + [1]      # the first frame after the pause is given up again
        i += k + 1
    assert _run(vsc, len(expect), at) == expect


def test_rare_ones_cost_64_frames_each(vsc):
    # ten launches given up, far apart: no pause grows
    n = 10 * 2000
    got = _run(vsc, n, range(0, n, 2000))
    assert [got[i:i + 2000].count(0) for i in range(0, n, 2000)] == [64] * 10


def test_pause_shrinks_with_resident_frames(vsc):
    # two in a row (128 frames), then 130 resident frames: the next one costs 128 again, not 256
    n = 1000
    got = _run(vsc, n, [0, 64, 64 + 128 + 130])
    assert got[:64] == [0] * 64 and got[64:192] == [0] * 128 and got[192:322] == [1] * 130
    assert got[322:450] == [0] * 128 and got[450:] == [1] * 550


def test_without_one_every_frame_is_resident(vsc):
    assert _run(vsc, 100, []) == [1] * 100
