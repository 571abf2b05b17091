"""Device bytes of a stream (host side): what vsc_stream_create allocates, the
resident solver's control words included."""
import pytest

CONTROL_WORDS = 66 << 10


@pytest.mark.parametrize("size", [(200, 120, 100, 60), (37, 29, 37, 29), (4, 4, 4, 4), (1279, 719, 640, 360),
                                  (1920, 1080, 1920, 1080)])
def test_footprint_is_the_whole_allocation(vsc, size):
    W, H, fw, fh = size
    piece = lambda w, h: -(-(3 * w * h * 4) // 256) * 256
    need = sum(8 * piece(W >> j, H >> j) for j in range(4) if W >> j >= 1 and H >> j >= 1)
    need += 2 * piece(W, H) if (fw, fh) != (W, H) else 0
    assert vsc.lib().vsc_stream_footprint(W, H, fw, fh) == need + CONTROL_WORDS
