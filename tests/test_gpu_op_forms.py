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


# widths and alignments that used to be copied first, both sides of the line between one and three
# displacements a block, hanging slots of 1 to 3 pixels, images too narrow for wide loads
@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("shape", [(1, 33, 16, 225), (1, 32, 20, 193), (1, 31, 29, 222), (2, 64, 9, 67), (1, 5, 3, 1),
                                   (1, 40, 5, 2), (2, 37, 6, 3), (1, 8, 2, 4), (1, 65, 37, 31)])
def test_correlation_lowp_reads_any_width(vsc, orc, cuda, kind, shape):
    """The bits of the same values in rows of a multiple of 4 (zeros to the
    right, as outside the image), and of operands one element off their
    alignment.  16-bit values also against the oracle: their products are exact
    in FP32, so only the FP32 sums of C terms round, and 2 C ulps of the sum of
    magnitudes bounds any order."""
    import torch
    N, C, H, W = shape
    rng = np.random.default_rng(sum(shape))
    f1, f2 = rng.standard_normal(shape).astype(np.float32), rng.standard_normal(shape).astype(np.float32)
    if kind == "fp8":
        q = [_t(rng.integers(0, 0x78, shape).astype(np.uint8), cuda) for _ in range(2)]
        one = torch.ones(1, device=cuda)
        call = lambda a, b: vsc.correlation_fp8(a, b, one, 4, 0)
    else:
        dt = torch.bfloat16 if kind == "bf16" else torch.float16
        q = [_t(x, cuda).to(dt) for x in (f1, f2)]
        call = lambda a, b: vsc.correlation(a, b, 4, 0)
    print(f"corr {kind} {shape}", flush=True)
    got = call(*q)
    off, wide = [], []
    for x in q:
        buf = torch.empty(x.numel() + 1, dtype=x.dtype, device=cuda)
        off.append(buf[1:].view(x.shape))
        off[-1].copy_(x)
        wide.append(torch.zeros((N, C, H, (W + 7) // 4 * 4), dtype=x.dtype, device=cuda))
        wide[-1][..., :W] = x
    assert torch.equal(call(*off), got)
    assert torch.equal(call(*wide)[..., :W], got)
    if kind != "fp8":
        f1, f2 = (x.float().cpu().numpy() for x in q)
        bound = orc.correlation(np.abs(f1), np.abs(f2), 4)
        assert np.all(np.abs(got.cpu().numpy() - orc.correlation(f1, f2, 4)) <= 2 * C * 2.0 ** -24 * bound + 1e-30)


@pytest.mark.parametrize("shape", [(2, 5, 3, 1), (1, 300, 7, 9), (1, 3, 67, 61), (3, 257, 4, 8), (1, 2, 257, 256)])
def test_fp8_quantiser_planes(vsc, cuda, shape):
    """Plane sizes around the quantiser's 4-pixel groups and 1024- and
    4096-pixel blocks, more channels than threads: the bits of the same
    formulas in FP32 (numpy), a channel of zeros among them."""
    import torch
    rng = np.random.default_rng(sum(shape))
    f1 = rng.standard_normal(shape).astype(np.float32)
    f2 = (rng.standard_normal(shape) * np.exp(rng.uniform(-2, 2, (1, shape[1], 1, 1)))).astype(np.float32)
    f1[:, 1] = 0
    m1, m2 = np.abs(f1).max(axis=(0, 2, 3)), np.abs(f2).max(axis=(0, 2, 3))
    r = np.where((m1 > 0) & (m2 > 0), np.sqrt(m2 / np.where(m1 > 0, m1, 1), dtype=np.float32), np.float32(1))
    s1, s2 = (m1 * r).max() / np.float32(448), (m2 / r).max() / np.float32(448)
    e = [(f1 * r[None, :, None, None]) / s1, (f2 / r[None, :, None, None]) / s2]
    q1, q2, sc = vsc.quantize_fp8_pair(_t(f1, cuda), _t(f2, cuda))
    for q, x in zip((q1, q2), e):
        assert torch.equal(q.cpu(), torch.from_numpy(x.astype(np.float32)).to(torch.float8_e4m3fn).view(torch.uint8))
    assert abs(float(sc.cpu()[0]) - float(s1 * s2)) <= 1e-6 * float(s1 * s2)
