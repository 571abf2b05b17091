"""Levels too large for the chip, swept in resident strips, against the blocked
solver (taken under graph capture) and the ticket form (after a launch that was
given up): the same operations for every pixel, so equal bit for bit, in any
order of routes between frames."""
import ctypes
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one round in two strips; several rounds with a shorter last one; odd sizes; strips of unequal height; reference order
@pytest.mark.parametrize("mode,W,H,levels,iters", [(2, 2304, 1000, 1, 40), (2, 2563, 1439, 2, 149), (2, 3001, 1301, 1, 101),
                                                   (2, 3840, 2160, 1, 31), (0, 2880, 2160, 1, 50)])
def test_strip_routes_agree(cuda, mode, W, H, levels, iters):
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    L = vsc.lib()
    out, xs, ys = (ctypes.c_int * 8)(), (ctypes.c_int * 1024)(), (ctypes.c_int * 1024)()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert not L.vsct_resident_plan(W, H, iters, cus, int(mode == 2), out, xs, ys)
    assert L.vsct_resident_strips(W, H, iters, cus, int(mode == 2), out, xs, ys)
    print(f"strips {(mode, W, H, levels, iters)}: {list(out)}", flush=True)
    n = 5
    g = torch.Generator(device="cuda").manual_seed(W + H)
    img = lambda: [torch.randint(0, 256, (H, W, 4), dtype=torch.uint8, device=cuda, generator=g) for _ in range(n)]
    o, p = img(), img()
    f = (torch.rand((H, W, 2), device=cuda, generator=g) * 6 - 3).contiguous()
    prm = vsc.HyperParams(pyramidLevels=levels, numIter=iters)
    L.vsct_resident_give_up.argtypes = [ctypes.c_void_p, ctypes.c_void_p]

    def sequence(route):
        st = vsc.VideoStabilizer(W, H, mode=mode)
        st.set_last_rgba(p[2])
        outs = []
        for t in range(1, n - 1):
            rgba = torch.zeros((H, W, 4), dtype=torch.uint8, device=cuda)
            of = torch.zeros((H, W, 3), device=cuda)
            step = lambda: st.do_one_step(o[t - 1:t + 2], p[t - 1:t + 2], f, f, out_rgba=rgba, out_float=of, params=prm)
            r = route(t)
            if r == "blocked":
                torch.cuda.synchronize()
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph):
                    step()
                graph.replay()
            else:
                if r == "ticket":
                    assert L.vsct_resident_give_up(st._h, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 1
                step()
            torch.cuda.synchronize()
            outs.append((rgba, of))
        st.close()
        return outs

    ref = sequence(lambda t: "blocked")
    for other in (sequence(lambda t: "strips"), sequence(lambda t: "ticket" if t == 1 else "strips"),
                  sequence(lambda t: "strips" if t % 2 else "blocked")):
        for (ra, fa), (rb, fb) in zip(ref, other):
            assert torch.equal(fa.view(torch.int32), fb.view(torch.int32)) and torch.equal(ra, rb)
