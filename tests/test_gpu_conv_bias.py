"""FP32 convolutions whose bias is read before or after the products, by the blocks
of their grid: the sums without a bias plus the bias, bit for bit."""
import pytest

pytestmark = pytest.mark.gpu


# grids of 640, 768, 769, 1020 and 1050 blocks of the 32-channel tile (stride 1: 8 x 16 pixels, stride 2: 4 x 16)
@pytest.mark.parametrize("shape", [(1, 256, 320, 32, 32, 1), (1, 384, 256, 32, 24, 1), (1, 386, 256, 16, 32, 1),
                                   (1, 272, 480, 32, 32, 1), (2, 200, 330, 64, 20, 1), (1, 360, 640, 32, 32, 2),
                                   (1, 216, 480, 16, 32, 2)])
def test_bias_early_or_late(vsc, cuda, shape):
    import torch
    import torch.nn.functional as F
    N, H, W, cin, cout, stride = shape
    print(f"conv bias {shape}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    x = torch.randn((N, H, W, cin), device=cuda, generator=g)
    w = torch.randn((cout, 3, 3, cin), device=cuda, generator=g) / (3 * cin ** 0.5)
    b = torch.randn(cout, device=cuda, generator=g)
    plain = vsc.conv3x3_nhwc(x, w, None, stride)
    # the same sums in the same order, and one rounding for the bias
    assert torch.equal(vsc.conv3x3_nhwc(x, w, torch.zeros(cout, device=cuda), stride), plain)
    assert torch.equal(vsc.conv3x3_nhwc(x, w, b, stride), plain + b)
    # a corner against 64 bits: 2 * 9 Cin roundings of the sum of magnitudes
    xs, ws = x[:1, :40, :40].permute(0, 3, 1, 2).double().cpu(), w.permute(0, 3, 1, 2).double().cpu()
    n = 18 // stride
    ref = F.conv2d(xs, ws, None, stride, 1)[..., :n, :n]
    mag = F.conv2d(xs.abs(), ws.abs(), None, stride, 1)[..., :n, :n]
    err = (plain[:1, :n, :n].permute(0, 3, 1, 2).double().cpu() - ref).abs()
    assert bool((err <= 2 * 9 * cin * 2.0 ** -24 * mag).all())
