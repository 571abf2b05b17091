"""The FP8 quantiser on more planes than one launch holds blocks (2^23): the same
formulas in FP32 on the host for the last item's channels and for the first one's."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(300, 60000, 1, 1), (180, 50000, 1, 3)])
def test_many_small_planes(vsc, cuda, shape):
    import torch
    print(f"fp8 planes {shape}", flush=True)
    g = torch.Generator().manual_seed(5)
    f1, f2 = torch.randn(shape, generator=g), torch.randn(shape, generator=g) * 3
    m1, m2 = (f.abs().amax(dim=(0, 2, 3)) for f in (f1, f2))
    r = torch.sqrt(m2 / m1)
    s1, s2 = (m1 * r).max() / 448, (m2 / r).max() / 448
    q1, q2, sc = vsc.quantize_fp8_pair(f1.to(cuda), f2.to(cuda))
    for n in (0, shape[0] // 2, shape[0] - 1):
        for q, e in ((q1, f1[n] * r[:, None, None] / s1), (q2, f2[n] / r[:, None, None] / s2)):
            assert torch.equal(q[n].cpu(), e.to(torch.float8_e4m3fn).view(torch.uint8)), n
