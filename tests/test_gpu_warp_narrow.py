"""Warp on maps narrower than a wave, whose rows share one: the bits of the same
map with columns added to the right (positions that stay inside the narrow map,
so that both read the same corners), at widths around the powers of two and rows
around a block's."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("N,C,H", [(1, 5, 1), (2, 4, 65), (1, 9, 130)])
@pytest.mark.parametrize("W", [1, 2, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65])
def test_narrow_maps_equal_wide_ones(vsc, cuda, dtype, N, C, H, W):
    import torch
    print(f"warp {dtype} {(N, C, H, W)}", flush=True)
    dt = getattr(torch, dtype)
    g = torch.Generator(device="cuda").manual_seed(W + H)
    x = torch.randn((N, C, H, W), device=cuda, generator=g, dtype=dt)
    # target columns in [0, W - 1], rows some of them outside
    to = torch.rand((N, 1, H, W), device=cuda, generator=g, dtype=dt) * (W - 1)
    f = torch.cat([to - torch.arange(W, device=cuda, dtype=dt), torch.randn((N, 1, H, W), device=cuda, generator=g, dtype=dt) * 3], 1)
    f[:, 0] = torch.where(f[:, 0] + torch.arange(W, device=cuda, dtype=dt) > W - 1, torch.zeros_like(f[:, 0]), f[:, 0])
    wide = 200
    xw, fw = torch.zeros((N, C, H, wide), device=cuda, dtype=dt), torch.zeros((N, 2, H, wide), device=cuda, dtype=dt)
    xw[..., :W], fw[..., :W] = x, f
    got, ref = vsc.warp(x, f.contiguous()), vsc.warp(xw, fw)[..., :W]
    # (a target on the last column has its right corner outside the narrow map and at weight 0 in the wide one)
    assert torch.equal(got, ref)
