"""FP32 Correlation on maps of one or two 8-pixel tiles across, whose form goes by
those tiles, around the lines between the forms: bit exact against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 17, 224, 5), (1, 9, 232, 8), (1, 21, 672, 4), (1, 5, 684, 7), (1, 3, 960, 8),
                                   (1, 3, 968, 6), (1, 33, 112, 9), (1, 6, 120, 16), (2, 5, 165, 13), (1, 4, 490, 16)])
@pytest.mark.parametrize("md", [1, 4])
def test_narrow_maps_bit_exact(vsc, orc, cuda, md, shape):
    import torch
    rng = np.random.default_rng(md + sum(shape))
    f1, f2 = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))
    print(f"corr f32 md={md} {shape}", flush=True)
    got = vsc.correlation(torch.from_numpy(f1).to(cuda), torch.from_numpy(f2).to(cuda), md, 0).cpu().numpy()
    assert np.array_equal(got, orc.correlation(f1, f2, md))
