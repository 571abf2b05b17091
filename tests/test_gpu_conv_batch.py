"""An item's result in a batch: layers of the flow network whose grid of eight
pairs would take other tiles than one pair's, and whole frames of four a call,
equal the ones computed alone bit for bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# H, W, Cin, Cout, dilation: decoder level 3 and refiner of an 854x480 frame (FP32) and of a 640x360 frame at half size
# (BF16); levels 4 and 5 of larger ones
@pytest.mark.parametrize("kind,shape", [("f32", (64, 112, 156, 128, 1)), ("f32", (64, 112, 256, 96, 1)),
                                        ("f32", (64, 112, 40, 128, 1)), ("f32", (96, 160, 160, 32, 1)),
                                        ("bf16", (24, 40, 256, 96, 1)), ("bf16", (24, 40, 256, 128, 1)),
                                        ("bf16", (48, 80, 160, 32, 1)), ("bf16", (24, 32, 128, 128, 1))])
def test_layer_items_equal_the_ones_alone(vsc, cuda, kind, shape):
    import torch
    H, W, Cin, Cout, dil = shape
    print(f"conv batch {kind} {shape}", flush=True)
    g = torch.Generator().manual_seed(sum(shape))
    dt, code = (torch.float32, 0) if kind == "f32" else (torch.bfloat16, 2)
    x = torch.randn((8, H, W, Cin), generator=g).to(dt).to(cuda)
    w = (torch.randn((Cout, 3, 3, Cin), generator=g) / (3 * Cin ** 0.5)).to(dt).contiguous()
    b = torch.randn(Cout, generator=g).to(cuda)
    P = lambda t: ctypes.c_void_p(t.data_ptr())

    def layer(inp):
        out = torch.zeros((inp.shape[0], H, W, Cout), dtype=dt, device=cuda)
        rc = vsc.lib().vsct_conv3x3_packed(P(inp), inp.shape[0], H, W, Cin, P(w), P(b), P(out), Cout, 1, dil, 1, code, code,
                                           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        return out

    whole = layer(x)
    for i in (0, 5):
        assert torch.equal(layer(x[i:i + 1].contiguous())[0], whole[i])


@pytest.mark.parametrize("form,W,H", [("chosen", 640, 360), ("plain", 854, 480)])
def test_four_frames_a_call_equal_one(vsc, cuda, form, W, H):
    import torch
    orig, proc, _, _ = vsc.synth_video(width=W, height=H, nframes=7, nblobs=60, motion=3.0, patch_size=16, seed=W)
    o, p = ([torch.from_numpy(np.ascontiguousarray(x)).to(cuda) for x in v] for v in (orig, proc))
    window = lambda t: (o[t - 1], o[t], o[t + 1], p[t - 1], p[t], p[t + 1])

    def run(batch):
        pipe = vsc.Pipeline(W, H, form=form, seed=7, flow_head_scale=0.05, flow_batch=batch)
        pipe.set_last_rgba(p[2])
        outs = []
        for t in range(1, 5, batch):
            ts = list(range(t, t + batch))
            of = [torch.empty((H, W, 3), device=cuda) for _ in ts]
            pipe.frames([window(i) for i in ts], t, out_float=of)
            outs += of
        torch.cuda.synchronize()
        pipe.close()
        return outs

    for a, b in zip(run(1), run(4)):
        assert torch.equal(a, b)
