"""Every form of the FP32 Correlation and of Warp at the edges of its range:
the smallest and largest grids of each tile, remainders of tiles, slots that
hang over the right edge, chunk remainders, images too narrow for wide loads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


# number of 32x8 tiles on both sides of the lines between the forms, odd widths, channels around a chunk
@pytest.mark.parametrize("shape", [(1, 65, 56, 31), (1, 64, 57, 29), (1, 41, 8, 670), (1, 1, 88, 64), (3, 21, 57, 33),
                                   (1, 17, 88, 130), (1, 16, 161, 183), (2, 33, 64, 225), (1, 5, 255, 255),
                                   (1, 9, 257, 249), (2, 4, 128, 256), (1, 6, 19, 4), (2, 7, 9, 3), (1, 4, 1, 6)])
@pytest.mark.parametrize("md", [0, 1, 3, 4])
def test_correlation_f32_forms_bit_exact(vsc, orc, cuda, md, shape):
    rng = np.random.default_rng(md * 100 + sum(shape))
    f1 = rng.standard_normal(shape).astype(np.float32)
    f2 = rng.standard_normal(shape).astype(np.float32)
    print(f"corr f32 md={md} {shape}", flush=True)
    got = vsc.correlation(_t(f1, cuda), _t(f2, cuda), md, 0).cpu().numpy()
    assert np.array_equal(got, orc.correlation(f1, f2, md))


@pytest.mark.parametrize("shape", [(1, 5, 6, 2), (2, 4, 3, 65), (1, 3, 5, 1), (1, 9, 2, 128)])
def test_warp_corners_at_the_edges(vsc, orc, cuda, shape):
    """Positions a hair outside each edge (mass inside above 0.999, so the pixel
    is kept with a corner missing), on the last column and row, and not finite.
    FP32 weights against the oracle's double ones: a few roundings of values
    of order 1."""
    N, C, H, W = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.uniform(-1, 1, shape).astype(np.float32)
    ys, xs = np.mgrid[0:H, 0:W].astype(np.float32)
    for tx, ty in ((-0.0005, 0), (W - 1 + 0.0005, 0), (0, -0.0005), (0, H - 1 + 0.0005), (W - 1, H - 1), (W - 1.5, 0),
                   (-1, 0), (W, 0), (np.inf, 0), (np.nan, 0)):
        fl = np.stack([np.stack([tx - xs, ty - ys])] * N).astype(np.float32)
        got = vsc.warp(_t(x, cuda), _t(fl, cuda)).cpu().numpy()
        assert np.max(np.abs(got - orc.warp(x, fl))) < 1e-5, (tx, ty)
