"""Frames on the default streams: the null stream (also while a blocking stream
is captured, when it cannot be asked for its own state) and the handle of the
per-thread one give the frame of an ordinary stream."""
import ctypes
import importlib

import pytest

pytestmark = pytest.mark.gpu

W, H = 320, 180


@pytest.fixture(scope="module")
def frame(cuda):
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    g = torch.Generator(device="cuda").manual_seed(3)
    img = lambda: [torch.randint(0, 256, (H, W, 4), dtype=torch.uint8, device=cuda, generator=g) for _ in range(3)]
    o, p = img(), img()
    f = (torch.rand((H, W, 2), device=cuda, generator=g) * 6 - 3).contiguous()
    fin = vsc.VscFrameIn(*(t.data_ptr() for t in (*o, *p, f, f)), 2)
    prm = vsc.HyperParams().c()
    keep = (o, p, f)

    def run(handle, around=None, mode=2):
        """Return code and frame of one call on the stream of this handle."""
        st = vsc.VideoStabilizer(W, H, mode=mode)
        st.set_last_rgba(keep[1][2])
        out = torch.zeros((H, W, 4), dtype=torch.uint8, device=cuda)
        torch.cuda.synchronize()
        call = lambda: vsc.lib().vsc_stab_frame(st._h, ctypes.byref(fin), ctypes.byref(prm), ctypes.c_void_p(out.data_ptr()),
                                                None, mode, ctypes.c_void_p(handle))
        rc = around(call) if around else call()
        torch.cuda.synchronize()
        st.close()
        return rc, out

    return run


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("handle", [0, 2])
def test_default_handles(cuda, frame, handle, mode):
    import torch
    rc, ref = frame(torch.cuda.Stream().cuda_stream, mode=mode)
    assert rc == 0
    rc, out = frame(handle, mode=mode)
    assert rc == 0 and torch.equal(out, ref)


@pytest.mark.parametrize("capture_mode", [0, 1, 2])
def test_legacy_stream_while_a_blocking_stream_is_captured(cuda, frame, capture_mode):
    import torch
    hip = ctypes.CDLL("libamdhip64.so.7")

    def captured(call):
        s, graph = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(s)) == 0
        assert hip.hipStreamBeginCapture(s, capture_mode) == 0
        rc = call()
        end = hip.hipStreamEndCapture(s, ctypes.byref(graph))
        hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(s)
        assert end == 0
        return rc

    rc, ref = frame(0)
    assert rc == 0
    rc, out = frame(0, captured)
    assert rc == 0 and torch.equal(out, ref)
