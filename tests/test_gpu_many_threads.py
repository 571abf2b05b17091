"""Calls that need more than 2^32 threads along a dimension of a launch: the FP32
Correlation of many maps less than 4 pixels wide (one thread an output), and Warp of
rows times channels beyond it.  Outputs of 20 and 17 GB."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def room(cuda):
    import torch
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 100 << 30:
        pytest.skip("needs 100 GB of free device memory")
    yield
    torch.cuda.empty_cache()


def test_correlation_of_many_narrow_maps(vsc, cuda, room):
    import torch
    N, H, W = 100, 200000, 3
    print("corr f32", (N, 1, H, W), flush=True)
    g = torch.Generator(device="cuda").manual_seed(2)
    a, b = (torch.randn((N, 1, H, W), device=cuda, generator=g) for _ in range(2))
    got = vsc.correlation(a, b, 4, 0)
    for n in (0, 57, N - 1):
        assert torch.equal(got[n], vsc.correlation(a[n:n + 1].contiguous(), b[n:n + 1].contiguous(), 4, 0)[0]), n


def test_warp_of_wide_rows_of_many_channels(vsc, cuda, room):
    import torch
    C, W = 65540, 65600
    print("warp f32", (1, C, 1, W), flush=True)
    x = torch.empty((1, C, 1, W), device=cuda)
    x[:] = torch.arange(C, device=cuda, dtype=torch.float32)[None, :, None, None]
    got = vsc.warp(x, torch.zeros((1, 2, 1, W), device=cuda))
    for c in range(0, C, 8192):
        assert torch.equal(got[:, c:c + 8192], x[:, c:c + 8192]), c
    assert torch.equal(got[:, -8:], x[:, -8:])
