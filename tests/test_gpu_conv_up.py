"""GPU: a doubling transposed convolution in one launch (conv_up) against its
four phases as offset-tap products (ien_multiply_ex)."""

import numpy as np
import pytest

from internal import conv_up

pytestmark = pytest.mark.gpu

TAPS = [[(0, 0)], [(0, 0), (0, 1)], [(0, 0), (1, 0)], [(0, 0), (0, 1), (1, 0), (1, 1)]]


def phases_of(ctx, c, n, rng):
    import ien

    bias = rng.standard_normal(n).astype(np.float32)
    return [ien.Matrix(ctx, (rng.standard_normal((len(t) * c, n)) / np.sqrt(len(t) * c)).astype(np.float32), bias)
            for t in TAPS]


def compare(ctx, x, h, w, c, n, phases, ys, act):
    import ien
    import torch

    y = torch.full((2 * h, 2 * w, ys), 7.0, dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()  # (the library's stream need not be torch's)
    conv_up(ctx, x, h, w, c, phases, y, ys, act)
    one = torch.empty((h, w, n), dtype=torch.float16, device="cuda")
    worst = 0.0
    for p, taps in enumerate(TAPS):
        ien.multiply_ex(ctx, ien.image_input(x, h, w, c, offsets=taps), 0, h * w, phases[p], one, n, act=act)
        torch.cuda.synchronize()
        got = y[p // 2::2, p % 2::2]
        for r in range(0, h, 256):  # (f32 copies of a band at a time)
            a, b = got[r:r + 256, :, :n].float(), one[r:r + 256].float()
            # f32 sums in another order: within 1e-5 of the terms' size, and
            # one f16 rounding (a spacing of 2^-10) either way.
            assert bool(((a - b).abs() <= 1e-5 + 2.0 ** -10 * b.abs()).all()), (p, r)
            worst = max(worst, float((a - b).abs().max()))
        torch.cuda.synchronize()  # (`one` is read)
        assert ys == n or bool((got[..., n:] == 7.0).all())
    print(f"  {h}x{w} {c}->{n}: {worst:.3g}", flush=True)


# Rows and columns about the 8 x 32 tiles, columns of outputs short of a 64,
# one and several chunks of channels, padded rows.
@pytest.mark.parametrize("h,w,c,n,pad,act", [
    (1, 1, 64, 8, 0, 0), (2, 3, 512, 256, 0, 1), (8, 32, 128, 64, 0, 1), (9, 33, 256, 128, 8, 1),
    (7, 31, 192, 72, 0, 0), (85, 125, 512, 256, 0, 1), (40, 200, 128, 64, 16, 2), (3, 65, 64, 16, 0, 4)])
def test_doubling_matches_its_phases(ctx, h, w, c, n, pad, act):
    import torch

    print(f"doubling {h}x{w} {c}->{n}", flush=True)
    rng = np.random.default_rng(h * w + c)
    x = torch.from_numpy(rng.standard_normal((h, w, c)).astype(np.float16)).cuda()
    compare(ctx, x, h, w, c, n, phases_of(ctx, c, n, rng), n + pad, act)


def test_doubling_refuses_prelu(ctx):
    import ien
    import torch

    rng = np.random.default_rng(2)
    x = torch.zeros((2, 2, 64), dtype=torch.float16, device="cuda")
    y = torch.zeros((4, 4, 8), dtype=torch.float16, device="cuda")
    with pytest.raises(ien.IenError) as e:
        conv_up(ctx, x, 2, 2, 64, phases_of(ctx, 64, 8, rng), y, 8, ien.ACT_PRELU)
    assert e.value.status == ien.ERR_INPUT


def test_doubling_of_the_largest_map(ctx):
    """The last doubling of a 6384 x 5256 image (33 554 304 padded pixels): an
    input of 2^31 - 2^13 bytes, outputs of 2^31 - 2^13 values."""
    import torch

    h, w, c, n = 5256 // 2, 6384 // 2, 128, 64
    print(f"doubling {h}x{w} {c}->{n}", flush=True)
    rng = np.random.default_rng(1)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.empty((h, w, c), dtype=torch.float16, device="cuda").normal_(generator=g)
    compare(ctx, x, h, w, c, n, phases_of(ctx, c, n, rng), n, 1)
    del x
    torch.cuda.empty_cache()
