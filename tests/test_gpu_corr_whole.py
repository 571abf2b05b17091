"""The reduced-precision Correlation with all vertical displacements in one block
(few channels, large maps) at the edges of its range: the bits of the same pixels
in a narrower map, which the other forms take (a pixel's sums depend on its
neighbourhood alone, in the same order in every form)."""
import pytest

pytestmark = pytest.mark.gpu


# 400 and 2500 tiles of 32 x 4 pixels and one fewer, 16 and 32 channels and one more, remainders of tiles, two items
@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("legacy", [0, 1])
@pytest.mark.parametrize("shape", [(1, 16, 64, 800), (1, 16, 61, 797), (1, 16, 60, 833), (1, 17, 64, 800), (2, 1, 33, 801),
                                   (1, 32, 200, 1600), (1, 31, 197, 1569), (1, 33, 200, 1600), (1, 32, 200, 1568)])
def test_whole_blocks_equal_the_other_forms(vsc, cuda, kind, legacy, shape):
    import torch
    N, C, H, W = shape
    print(f"corr {kind} {shape} legacy={legacy}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    if kind == "fp8":
        f = [torch.randint(0, 0x78, shape, dtype=torch.uint8, device=cuda, generator=g) for _ in range(2)]
        one = torch.ones(1, device=cuda)
        call = lambda a, b: vsc.correlation_fp8(a, b, one, 4, legacy)
    else:
        dt = torch.bfloat16 if kind == "bf16" else torch.float16
        f = [torch.randn(shape, device=cuda, generator=g).to(dt) for _ in range(2)]
        call = lambda a, b: vsc.correlation(a, b, 4, legacy)
    got = call(*f)
    first = call(*(x[..., :100].contiguous() for x in f))          # 96 columns and the displacements' reach
    last = call(*(x[..., W - 100:].contiguous() for x in f))
    assert torch.equal(got[..., :96], first[..., :96])
    assert torch.equal(got[..., W - 96:], last[..., 4:])


# fewer displacements: one a block up to 512 blocks, all of them above (73, 102 and 170 tiles); the columns come from a
# map of 36 tiles, which takes one a block
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
@pytest.mark.parametrize("md", [0, 1, 2, 3])
@pytest.mark.parametrize("shape", [(1, 40, 33, 257), (1, 9, 36, 256), (2, 33, 36, 290), (1, 65, 36, 640)])
def test_fewer_displacements(vsc, cuda, kind, md, shape):
    import torch
    N, C, H, W = shape
    print(f"corr {kind} md={md} {shape}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(shape) + md)
    if kind == "fp8":
        f = [torch.randint(0, 0x78, shape, dtype=torch.uint8, device=cuda, generator=g) for _ in range(2)]
        one = torch.ones(1, device=cuda)
        call = lambda a, b: vsc.correlation_fp8(a, b, one, md, 0)
    else:
        f = [torch.randn(shape, device=cuda, generator=g).to(torch.bfloat16) for _ in range(2)]
        call = lambda a, b: vsc.correlation(a, b, md, 0)
    got = call(*f)
    assert torch.equal(got[:1, ..., :96], call(*(x[:1, ..., :100].contiguous() for x in f))[..., :96])
