"""The sizes that the convolution kernels accept (host code, no GPU)."""

import pytest

from internal import conv_up_fits


# LaMa's maps at P padded pixels: 64 channels at full scale, 128, 256 and 512
# at the levels below.  The first convolution writes P x 64 values and takes
# them in 31 bits, so every P below 2^25 (a multiple of 64) has to come up
# through the three doublings; the next one is refused by both.
@pytest.mark.parametrize("pixels,fits", [
    (256, True), (2 ** 25 - 2 ** 10, True), (6384 * 5256, True), (2 ** 25 - 64, True), (2 ** 25, False)])
def test_doublings_take_every_map_that_fits_the_first_convolution(pixels, fits):
    levels = [(512, 256), (256, 128), (128, 64)]
    assert all(conv_up_fits(1, pixels // 64 * 4 ** i, c, n, n) for i, (c, n) in enumerate(levels)) == fits


@pytest.mark.parametrize("h,w,c,n,ys", [(0, 4, 64, 64, 64), (4, 4, 48, 64, 64), (4, 4, 64, 60, 64),
                                        (4, 4, 64, 64, 56), (4, 4, 64, 64, 68)])
def test_doublings_refuse_other_layouts(h, w, c, n, ys):
    assert not conv_up_fits(h, w, c, n, ys)
