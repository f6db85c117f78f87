"""The sizes that the convolution, chain and row-product kernels accept, and
which of them a size takes (host code, no GPU)."""

import pytest

from internal import chain_choice, conv3_choice, conv_up_fits, rows_choice, stride2_choice

CUS, WORKSPACE = 256, 8 << 20  # MI355X; the context's workspace in floats


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


# conv_wide's tiles in order: 8 x 64, 4 x 128, 8 x 128, 4 x 64 (rows x
# channels, 32 pixels wide).  The sizes of test_gpu_conv's test_conv3x3_wide
# and its splits, which are there for the tile named here.
@pytest.mark.parametrize("h,w,c,n,row0,rows,want", [
    (85, 125, 512, 128, 0, None, (3, 1)), (61, 67, 384, 136, 0, None, (3, 1)), (70, 77, 512, 128, 0, None, (0, 4)),
    (95, 95, 512, 232, 0, None, (1, 1)), (131, 163, 128, 200, 0, None, (2, 1)), (253, 250, 128, 64, 700, 62001, (0, 1)),
    (2, 4000, 512, 128, 0, None, (3, 1)), (2500, 3, 192, 128, 0, None, (1, 1)),
    (40, 200, 512, 128, 0, None, (1, 3)), (73, 200, 768, 120, 0, None, (2, 3)), (49, 200, 1024, 128, 0, None, (1, 2)),
    (64, 64, 512, 128, 0, None, None)])
def test_wide_tiles(h, w, c, n, row0, rows, want):
    assert conv3_choice(CUS, WORKSPACE, w, c, n, row0, row0 + (h * w if rows is None else rows)) == want


# A band of a tall map is the work of a map of its own height: 4 rows of 1000 x
# 64 pixels, 512 -> 128, took 15.0 us on the tiles that suit the whole map, 10.2
# on the general kernel's splits.
@pytest.mark.parametrize("w,c,n", [(64, 512, 128), (95, 512, 256), (125, 512, 128), (300, 256, 256), (512, 128, 128)])
@pytest.mark.parametrize("first,rows", [(0, 4), (8, 4), (480, 8), (96, 20), (16, 40), (800, 100)])
def test_bands_choose_by_their_own_rows(w, c, n, first, rows):
    assert conv3_choice(CUS, WORKSPACE, w, c, n, first * w, (first + rows) * w) == \
        conv3_choice(CUS, WORKSPACE, w, c, n, 0, rows * w)


def test_a_narrow_band_keeps_the_general_kernels_splits():
    assert conv3_choice(CUS, WORKSPACE, 64, 512, 128, 500 * 64, 504 * 64) is None
    assert conv3_choice(CUS, WORKSPACE, 64, 512, 128, 0, 1000 * 64) is not None


# Stride 2 the same: 16 rows of a 256 x 256 output, 256 -> 512, took 20.8 us on
# the whole map's 16-channel chunks, 17.9 on 32-channel ones.
def test_stride2_bands_choose_by_their_own_rows():
    assert stride2_choice(CUS, 256, 512, 0, 256 * 256) == 16
    assert stride2_choice(CUS, 256, 512, 100 * 256, 116 * 256) == 32
    assert stride2_choice(CUS, 256, 512, 0, 16 * 256) == 32
    # 256 tiles are a CU's each, one more is not.
    assert stride2_choice(CUS, 256, 64, 0, 128 * 256) == 32
    assert stride2_choice(CUS, 256, 64, 0, 128 * 256 + 1) == 16
    assert stride2_choice(CUS, 256, 64, 2 * 256, 130 * 256) == 16


# Products of few channels and 96 tiles or more keep four waves a tile: eight
# lose on three 64-deep chunks and less (3951 x 64 -> 192 4.2 us on four, 4.7 on
# eight).
@pytest.mark.parametrize("m,n", [(96 * 64, 128), (1762, 520), (3951, 192), (8000, 256), (8192, 256)])
def test_shallow_products_keep_four_waves(m, n):
    for k in (64, 128, 192):
        assert rows_choice(CUS, WORKSPACE, m, k, n) == (4, 1)
    for k in (256, 384, 448):
        assert rows_choice(CUS, WORKSPACE, m, k, n) == (8, 1)
    assert rows_choice(CUS, WORKSPACE, m, 288, n) == (4, 1)  # (not whole 64-deep chunks)


@pytest.mark.parametrize("m,n", [(1, 8), (900, 128), (95 * 64, 128)])
def test_shallow_products_of_few_tiles_take_eight_waves(m, n):
    for k in (64, 128, 192, 256):
        assert rows_choice(CUS, WORKSPACE, m, k, n) == (8, 1)
    assert rows_choice(CUS, WORKSPACE, m, 96, n) == (4, 1)


def test_more_tiles_than_cus_keep_four_waves():
    assert rows_choice(CUS, WORKSPACE, 8193, 384, 256) == (4, 1)
    assert rows_choice(CUS, WORKSPACE, 64 * 257, 1536, 128) == (4, 1)
    assert rows_choice(CUS, WORKSPACE, 128 * 128, 1536, 64) == (4, 1)  # 128-row tiles


# Deep products of few tiles: split where a tile a CU in one launch would take
# longer (4600 x 3392 -> 24 15.5 us split, 18.9 in one; 4500 x 3104 -> 24, which
# four waves take, 14.7 and 25.4), and in one launch where the sums cost more
# (2319 x 1664 -> 584 13.5 us in one, 21.2 split).
@pytest.mark.parametrize("m,k,n,want", [
    (4600, 3392, 24, (4, 8)), (3200, 2560, 24, (4, 10)), (3256, 1728, 8, (4, 6)), (4100, 4096, 24, (4, 8)),
    (2300, 4096, 200, (4, 8)), (4500, 3104, 24, (4, 8)), (1100, 2080, 512, (4, 8)), (100, 4096, 256, (4, 16)),
    (2319, 1664, 584, (8, 1)), (4600, 1536, 64, (8, 1)), (4096, 1536, 384, (8, 1)), (949, 2048, 512, (8, 1)),
    (2000, 1568, 512, (4, 1)), (16500, 1536, 64, (4, 1))])
def test_deep_products_split_where_that_is_faster(m, k, n, want):
    assert rows_choice(CUS, WORKSPACE, m, k, n) == want


def test_splits_stay_in_the_workspace():
    for m in (100, 700, 2300, 4600, 8000):
        for k in (1536, 2560, 4096):
            for n in (8, 64, 200, 512):
                for workspace in (1 << 14, 1 << 20, WORKSPACE):
                    waves, splits = rows_choice(CUS, workspace, m, k, n)
                    assert splits == 1 or splits * m * ((n + 127) // 128 * 128) <= workspace


# A chain's workgroups wait for each other, so all of them have to be resident:
# the chains of small maps on smaller tiles take a quarter of the CUs at most,
# so that the four streams that a process runs at once hold one each, as they
# did on 16 x 24 tiles.
@pytest.mark.parametrize("h,w,want", [
    (1, 1, (8, 16)), (48, 64, (8, 16)), (64, 128, (8, 16)), (65, 128, (12, 16)), (72, 160, (12, 16)),
    (96, 128, (12, 16)), (97, 128, (16, 24)), (128, 128, (16, 24)), (128, 256, (16, 24)), (192, 256, (16, 24)),
    (256, 384, (16, 24)), (257, 384, None), (256, 385, None), (8, 1024, (8, 16)), (8, 1025, (16, 24))])
def test_chain_tilings(h, w, want):
    assert chain_choice(CUS, h, w) == want


def test_four_chains_that_fitted_on_large_tiles_fit():
    for h in range(1, 400, 3):
        for w in range(1, 500, 7):
            large = ((h + 15) // 16) * ((w + 23) // 24)
            tile = chain_choice(CUS, h, w)
            assert (tile is None) == (large > CUS)
            if tile:
                tiles = -(-h // tile[0]) * -(-w // tile[1])
                for streams in (1, 2, 3, 4):
                    assert streams * large > CUS or streams * tiles <= CUS
