"""Few sweeps of a large level, swept in resident strips, against the blocked
solver (taken under graph capture): with a large step a value that a strip's cut
makes wrong would still weigh half a unit in the last place after 12 sweeps.
The same operations for every pixel, so equal bit for bit."""
import ctypes
import importlib

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,W,H,iters", [(2, 3840, 2160, 12), (2, 2560, 1440, 12), (0, 3840, 2160, 16)])
def test_few_sweeps_in_strips(cuda, mode, W, H, iters):
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    L = vsc.lib()
    out, xs, ys = (ctypes.c_int * 8)(), (ctypes.c_int * 1024)(), (ctypes.c_int * 1024)()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert L.vsct_resident_strips(W, H, iters, cus, int(mode == 2), out, xs, ys)
    print(f"strips {(mode, W, H, iters)}: {list(out)}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(W + iters)
    img = lambda: [torch.randint(0, 256, (H, W, 4), dtype=torch.uint8, device=cuda, generator=g) for _ in range(3)]
    o, p = img(), img()
    f = (torch.rand((H, W, 2), device=cuda, generator=g) * 6 - 3).contiguous()
    prm = vsc.HyperParams(pyramidLevels=1, numIter=iters, stepSize=0.24, gamma=0.1)

    def frame(captured):
        st = vsc.VideoStabilizer(W, H, mode=mode)
        st.set_last_rgba(p[2])
        of = torch.zeros((H, W, 3), device=cuda)
        step = lambda: st.do_one_step(o, p, f, f, out_float=of, params=prm)
        if captured:
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                step()
            graph.replay()
        else:
            step()
        torch.cuda.synchronize()
        st.close()
        return of

    a, b = frame(False), frame(True)
    assert torch.isfinite(b).all()
    assert torch.equal(a.view(torch.int32), b.view(torch.int32)), int((a != b).sum())
