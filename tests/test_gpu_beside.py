"""Stabilizers that run side by side on HIP streams of their own.  A small frame
leaves most of the device idle in the resident solver, whose launches take turns,
so beside other stabilizers' frames it takes the blocked one; alone, on the same
HIP stream, and where the frame fills the device, it stays resident.  Frames are
the same bits either way."""
import importlib

import pytest

pytestmark = pytest.mark.gpu


class Stab:
    def __init__(self, vsc, cuda, W, H, mode, stream):
        import torch
        g = torch.Generator(device="cuda").manual_seed(W + H)
        img = lambda: [torch.randint(0, 256, (H, W, 4), dtype=torch.uint8, device=cuda, generator=g) for _ in range(3)]
        self.o, self.p = img(), img()
        self.f = (torch.rand((H, W, 2), device=cuda, generator=g) * 6 - 3).contiguous()
        self.vsc, self.stream = vsc, stream
        self.st = vsc.VideoStabilizer(W, H, mode=mode)
        self.st.set_last_rgba(self.p[2])
        self.out = torch.zeros((H, W, 4), dtype=torch.uint8, device=cuda)

    def frame(self):
        """The levels of the frame that were solved resident."""
        import torch
        with torch.cuda.stream(self.stream):
            self.st.do_one_step(self.o, self.p, self.f, self.f, out_rgba=self.out)
        return self.vsc.lib().vsct_resident_levels(self.st._h)


@pytest.mark.parametrize("mode,small", [(2, (320, 180)), (0, (320, 180)), (2, (640, 360))])
def test_small_frames_beside_others_are_blocked(cuda, mode, small):
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    a = Stab(vsc, cuda, 1920, 1080, 2, torch.cuda.Stream())
    b = Stab(vsc, cuda, *small, mode, torch.cuda.Stream())
    ref = Stab(vsc, cuda, *small, mode, b.stream)
    torch.cuda.synchronize()
    assert a.frame() == 2
    torch.cuda.synchronize()
    assert b.frame() == 2          # nothing is under way
    torch.cuda.synchronize()
    for _ in range(40):            # some 20 ms of frames
        a.frame()
    assert b.frame() == 0
    assert a.frame() == 2          # a frame that fills the device stays resident
    torch.cuda.synchronize()
    for _ in range(64):
        b.frame()
        torch.cuda.synchronize()
    assert b.frame() == 2          # and the small one is again, once it is alone
    torch.cuda.synchronize()
    for _ in range(67):
        ref.frame()
        torch.cuda.synchronize()
    assert torch.equal(b.out, ref.out)
    for s in (a, b, ref):
        s.st.close()


def test_stabilizers_on_one_stream_stay_resident(cuda):
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    s = torch.cuda.Stream()
    a, b = Stab(vsc, cuda, 1920, 1080, 2, s), Stab(vsc, cuda, 320, 180, 2, s)
    torch.cuda.synchronize()
    for _ in range(10):
        assert a.frame() == 2 and b.frame() == 2
    torch.cuda.synchronize()
    a.st.close()
    b.st.close()


@pytest.mark.parametrize("threads", [False, True])
@pytest.mark.parametrize("capture_mode", [0, 1, 2])
def test_asking_for_others_leaves_a_capture_whole(cuda, capture_mode, threads):
    """The frames' marks and queries while a third stream is captured, by the thread
    that captures and by another."""
    import ctypes
    import threading
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    hip = ctypes.CDLL("libamdhip64.so.7")
    a = Stab(vsc, cuda, 1920, 1080, 2, torch.cuda.Stream())
    b = Stab(vsc, cuda, 320, 180, 2, torch.cuda.Stream())
    ref = Stab(vsc, cuda, 320, 180, 2, b.stream)
    torch.cuda.synchronize()
    for s in (a, b):
        s.frame()
    torch.cuda.synchronize()
    c, graph = torch.cuda.Stream(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(ctypes.c_void_p(c.cuda_stream), capture_mode) == 0

    def frames():
        for _ in range(10):
            a.frame()
            b.frame()

    try:
        if threads:
            t = threading.Thread(target=frames)
            t.start()
            t.join()
        else:
            frames()
    finally:
        end = hip.hipStreamEndCapture(ctypes.c_void_p(c.cuda_stream), ctypes.byref(graph))
        hip.hipGraphDestroy(graph)
    assert end == 0
    torch.cuda.synchronize()
    for _ in range(11):
        ref.frame()
        torch.cuda.synchronize()
    assert torch.equal(b.out, ref.out)
    for s in (a, b, ref):
        s.st.close()
