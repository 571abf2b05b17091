"""The resident consistency solver against the other routes of a frame: the
blocked solver (taken under graph capture) and the ticket form (taken when the
device cannot hold a resident launch).  All three compute every sweep of every
pixel with the same operations, so frames and RGBA8 outputs are equal bit for
bit, and a sequence may change routes between frames."""
import ctypes
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _video(vsc, cuda, W, H, n):
    import torch
    o, p, f, b = vsc.synth_video(width=W, height=H, nframes=n, nblobs=60, motion=3.0, patch_size=16, seed=W * 7 + H)
    return [[torch.from_numpy(np.ascontiguousarray(x)).to(cuda) for x in v] for v in (o, p, f, b)]


def _give_up(vsc, st):
    import torch
    L = vsc.lib()
    L.vsct_resident_give_up.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    assert L.vsct_resident_give_up(st._h, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 1


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("W,H,levels,iters", [(128, 48, 1, 20), (129, 49, 1, 19), (131, 65, 2, 33), (256, 64, 1, 8),
                                              (258, 98, 2, 75), (515, 201, 3, 100), (640, 360, 2, 150), (1282, 718, 2, 41),
                                              # one pixel a lane: levels one tile large, a pixel larger, flush on both sides
                                              (64, 64, 1, 21), (65, 67, 1, 40), (130, 66, 2, 150), (199, 113, 2, 33), (321, 181, 1, 26)])
def test_routes_agree(cuda, mode, W, H, levels, iters):
    """Tile edges and remainders (levels one tile large, one pixel larger, odd
    ones), whole and part phases, one to three levels, both solver forms."""
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    n = 6
    o, p, f, b = _video(vsc, cuda, W, H, n)
    prm = vsc.HyperParams(pyramidLevels=levels, numIter=iters)

    def sequence(route):
        st = vsc.VideoStabilizer(W, H, mode=mode)
        st.set_last_rgba(p[2])
        outs = []
        for t in range(1, n - 1):
            rgba = torch.zeros((H, W, 4), dtype=torch.uint8, device=cuda)
            of = torch.zeros((H, W, 3), device=cuda)
            step = lambda: st.do_one_step(o[t - 1:t + 2], p[t - 1:t + 2], f[t], b[t], out_rgba=rgba, out_float=of, params=prm)
            r = route(t)
            if r == "blocked":
                torch.cuda.synchronize()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g):
                    step()
                g.replay()
            else:
                if r == "ticket":
                    _give_up(vsc, st)
                step()
            torch.cuda.synchronize()
            outs.append((rgba.cpu().numpy(), of.cpu().numpy()))
        st.close()
        return outs

    ref = sequence(lambda t: "blocked")
    got = sequence(lambda t: "resident")
    # a given-up launch (then the blocked solver for the frames behind it), and routes in turn
    gave_up = sequence(lambda t: "ticket" if t == 1 else "resident")
    mixed = sequence(lambda t: "resident" if t % 2 else "blocked")
    for other in (got, gave_up, mixed):
        for (ra, fa), (rb, fb) in zip(ref, other):
            assert np.array_equal(fa, fb) and np.array_equal(ra, rb)


def test_two_streams_take_turns(cuda):
    """Two stabilizers driven on two HIP streams without synchronisation in
    between: each sequence equals the one computed alone."""
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    W, H, n = 640, 360, 8
    o, p, f, b = _video(vsc, cuda, W, H, n)

    def drive(st, out, t):
        st.do_one_step(o[t - 1:t + 2], p[t - 1:t + 2], f[t], b[t], out_rgba=out[t])

    buf = lambda: [torch.zeros((H, W, 4), dtype=torch.uint8, device=cuda) for _ in range(n)]
    ref = buf()
    st = vsc.VideoStabilizer(W, H, mode=vsc.VSC_FRAME_FMA)
    st.set_last_rgba(p[2])
    for t in range(1, n - 1):
        drive(st, ref, t)
    torch.cuda.synchronize()
    st.close()
    streams = [torch.cuda.Stream() for _ in range(2)]
    sts, outs = [], []
    for s in streams:
        with torch.cuda.stream(s):
            a = vsc.VideoStabilizer(W, H, mode=vsc.VSC_FRAME_FMA)
            a.set_last_rgba(p[2])
        sts.append(a)
        outs.append(buf())
    torch.cuda.synchronize()
    for t in range(1, n - 1):
        for s, a, out in zip(streams, sts, outs):
            with torch.cuda.stream(s):
                drive(a, out, t)
    torch.cuda.synchronize()
    for out in outs:
        for t in range(1, n - 1):
            assert torch.equal(out[t], ref[t])
    for a in sts:
        a.close()
