"""Upsampler gradients at the edges of the weight-gradient tiles (16 x 16
pixels) and of the reduction over tiles (32 rows at a time)."""
import importlib

import numpy as np
import pytest

from oracle import upsampler as ou

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,W,H", [(1, 6, 5), (1, 16, 16), (1, 17, 33), (3, 31, 15), (2, 64, 65), (5, 49, 50)])
def test_gradients_ragged_tiles(cuda, B, W, H):
    """Loss and gradient against the float64 oracle.  1 tile to 100 (33 and 45
    rows of partial sums: not whole groups of 32), tiles with 1 to 16 valid
    rows and columns.  Every gradient sum has 3*16 + 1 or fewer FP32 rounding
    steps of relative size 2^-24 per level over at most B*W*H pixel terms whose
    absolute sum the oracle's gradient bounds only with cancellation, so the
    bound is relative to the largest gradient of the layer."""
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    rng = np.random.default_rng(W * 100 + H)
    lo = rng.uniform(-3, 3, (B, (H + 1) // 2, (W + 1) // 2, 2)).astype(np.float32)
    fr = rng.integers(0, 256, (B, H, W, 4), dtype=np.uint8)
    gt = rng.uniform(-6, 6, (B, H, W, 2)).astype(np.float32)
    p = (0.2 * rng.standard_normal(vsc.Upsampler.param_count())).astype(np.float32)
    ups = vsc.Upsampler(params=p)
    T = lambda a: torch.from_numpy(a).to(cuda)
    loss, g = ups.loss_grad(T(lo), T(fr), T(gt))
    ref_loss, ref = ou.loss_and_grad(p, lo, fr, gt)
    assert abs(loss - ref_loss) <= 1e-5 * ref_loss
    o = 0
    for shape in ou.SHAPES:
        n = int(np.prod(shape))
        a, b = g[o:o + n].astype(np.float64), ref[o:o + n]
        assert np.max(np.abs(a - b)) <= 1e-4 * np.max(np.abs(ref)), shape
        o += n
    ups.close()
