"""How a packed layer groups its sums over input channels (host side): by one
batch item's geometry, so that an item has the same bits in a batch of any size."""
import pytest

# the flow network's decoder and refiner layers: input channels, output channels, stride, dilation
LAYERS = [(196, 196, 1, 1), (128, 196, 2, 1), (64, 64, 1, 1), (32, 64, 2, 1), (288, 128, 1, 1), (128, 128, 1, 1),
          (256, 128, 1, 1), (256, 96, 1, 1), (224, 64, 1, 1), (160, 32, 1, 1), (448, 2, 1, 1), (40, 128, 1, 1),
          (128, 128, 1, 2), (128, 128, 1, 4), (128, 96, 1, 8), (96, 64, 1, 16)]


@pytest.mark.parametrize("dtype", [0, 2])
def test_grouping_is_the_same_in_any_batch(vsc, dtype):
    flush = vsc.lib().vsct_conv_flush
    split = 0
    for H in list(range(1, 40, 3)) + list(range(40, 300, 17)):
        for W in list(range(1, 40, 5)) + list(range(40, 500, 23)):
            for layer in LAYERS:
                got = {flush(n, H, W, *layer, dtype) for n in range(1, 9)}
                assert len(got) == 1, (H, W, layer, got)
                split += got != {0}
    assert split > 1000
    # a layer of the FP32 network of an 854x480 frame and one of the BF16 network of a 640x360 frame at half size
    assert flush(1, 64, 112, 156, 128, 1, 1, 0) == flush(8, 64, 112, 156, 128, 1, 1, 0)
    assert flush(1, 24, 40, 256, 96, 1, 1, 2) == flush(6, 24, 40, 256, 96, 1, 1, 2)
