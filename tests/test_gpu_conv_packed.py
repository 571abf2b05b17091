"""Convolutions with packed weights (the flow network's layers) against FP64:
tile remainders in rows, columns and channels, channel tails of a K step,
dilation sub-grids smaller than a tile, stride 2, grids small enough to keep
their sums in parts and large enough for the tallest tiles.

Bound: products of the element types are exact in FP32 or rounded once, and
9 Cin terms are summed in FP32 in some order: 2 * 9 Cin * 2^-24 of the sum of
magnitudes, plus half an ulp (2^-9, doubled for the order of roundings) of a
BF16 output."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# N, H, W, Cin, Cout, stride, dilation
SHAPES = [(1, 1, 1, 24, 32, 1, 1), (2, 5, 3, 280, 128, 1, 1), (1, 9, 17, 40, 2, 1, 1), (2, 18, 31, 104, 96, 1, 1),
          (1, 16, 16, 32, 36, 1, 1), (1, 23, 40, 64, 64, 1, 16), (2, 33, 47, 48, 128, 1, 3), (1, 19, 35, 32, 64, 2, 1),
          (1, 64, 64, 24, 28, 2, 1), (1, 130, 100, 40, 160, 1, 1), (2, 72, 120, 32, 96, 1, 2), (1, 200, 330, 24, 64, 1, 1),
          (1, 40, 60, 200, 20, 1, 1), (1, 3, 50, 128, 16, 1, 1)]


@pytest.mark.parametrize("kind", ["f32", "bf16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_packed_layers_against_float64(vsc, cuda, kind, shape):
    import torch
    import torch.nn.functional as F
    N, H, W, Cin, Cout, st, dil = shape
    print(f"packed conv {kind} {shape}", flush=True)
    g = torch.Generator().manual_seed(sum(shape))
    dt, code = (torch.float32, 0) if kind == "f32" else (torch.bfloat16, 2)
    out_code, odt = (code, dt) if Cout > 16 else (0, torch.float32)   # the flow heads write FP32
    x = torch.randn((N, H, W, Cin), generator=g).to(dt)
    w = (torch.randn((Cout, 3, 3, Cin), generator=g) / (3 * Cin ** 0.5)).to(dt)
    b = torch.randn(Cout, generator=g)
    out = torch.full((N, (H - 1) // st + 1, (W - 1) // st + 1, Cout), 7.0, dtype=odt, device=cuda)
    xd, bd = x.to(cuda), b.to(cuda)
    L = vsc.lib()
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = L.vsct_conv3x3_packed(P(xd), N, H, W, Cin, P(w.contiguous()), P(bd), P(out), Cout, st, dil, 1, code, out_code,
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    xx, ww = x.double().permute(0, 3, 1, 2), w.double().permute(0, 3, 1, 2)
    ref = F.leaky_relu(F.conv2d(xx, ww, b.double(), st, dil, dil), 0.1)
    mag = F.conv2d(xx.abs(), ww.abs(), b.double().abs(), st, dil, dil)
    bound = 2 * (9 * Cin + 2) * 2.0 ** -24 * mag
    if odt == torch.bfloat16:
        bound = bound + 2.0 ** -8 * (ref.abs() + bound)
    err = (out.cpu().double().permute(0, 3, 1, 2) - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


def test_packed_weights_are_refused_where_they_do_not_fit(vsc, cuda):
    import torch
    x = torch.zeros((1, 8, 8, 16), dtype=torch.bfloat16, device=cuda)
    w = torch.zeros((32, 3, 3, 16), dtype=torch.bfloat16)
    out = torch.zeros((1, 8, 8, 32), dtype=torch.bfloat16, device=cuda)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    assert vsc.lib().vsct_conv3x3_packed(P(x), 1, 8, 8, 16, P(w), None, P(out), 32, 1, 1, 1, 2, 2, None) != 0
