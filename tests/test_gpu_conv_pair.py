"""GPU: the body kernels' tilings give the bits of single-layer launches.

ien_conv3_pair cuts a map into strips of 62 or 30 columns by segments of
rows, ien_conv3_chain into 8 x 16 or 12 x 16 tiles where they take at most a
quarter of the 256 CUs and else into 16 x 24 tiles, a CU each at most.  Both are compared, bit for bit, with one
ien_conv3 launch per layer at the edges of those cuts."""

import numpy as np
import pytest

import synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layers(ctx):
    import ien
    import torch

    host = synthetic.esrgan_layers(synthetic.esrgan_tensors())[1:5]
    # PReLU slopes of both signs, so that no layer is an identity.
    rng = np.random.default_rng(4)
    return [(ien.Matrix(ctx, w, b), torch.from_numpy(rng.uniform(-0.5, 1.2, 64).astype(np.float32)).cuda())
            for w, b, _ in host]


def single(ctx, x, h, w, layers):
    import ien
    import torch

    for m, slope in layers:
        y = torch.empty_like(x)
        ien.conv3(ctx, ien.image_input(x, h, w, 64), m, y, 64, finish=ien.ACT_PRELU, slope=slope)
        x = y
    return x


def same_bits(a, b):
    import torch

    torch.cuda.synchronize()  # the library's stream need not be torch's
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


# One column or row; widths on either side of a 30- and a 62-column strip;
# one segment a row and several rounds of workgroups; segments of unequal
# height; more strips than CUs.
@pytest.mark.parametrize("h,w", [(1, 1), (1, 200), (200, 1), (2, 30), (3, 31), (5, 62), (17, 63), (64, 125),
                                 (300, 500), (97, 1300), (3, 16400)])
def test_pair_strips(ctx, layers, h, w):
    import ien
    import torch

    print(f"pair {h}x{w}", flush=True)
    x = torch.from_numpy(np.random.default_rng(h * w).standard_normal((h, w, 64)).astype(np.float16)).cuda()
    y = torch.full_like(x, 7.0)
    torch.cuda.synchronize()
    (m1, s1), (m2, s2) = layers[:2]
    ien.conv3_pair(ctx, x, y, h, w, m1, s1, m2, s2)
    assert same_bits(y, single(ctx, x, h, w, layers[:2]))


# Both sides of the smaller tilings' 64 tiles (8 x 16 up to 64 x 128 pixels,
# 12 x 16 up to 96 x 128) and of 256 tiles of 16 x 24, partial tiles on both
# edges, last tiles narrower than the 2-pixel border.
@pytest.mark.parametrize("h,w", [(1, 1), (9, 17), (7, 100), (128, 256), (129, 256), (121, 273), (192, 256),
                                 (193, 256), (181, 273), (256, 384), (241, 361), (64, 128), (65, 128), (57, 113),
                                 (96, 128), (97, 128), (85, 113), (61, 161), (8, 1009), (1, 1025)])
def test_chain_tilings(ctx, layers, h, w):
    import ien
    import torch

    print(f"chain {h}x{w}", flush=True)
    x = torch.from_numpy(np.random.default_rng(h + w).standard_normal((h, w, 64)).astype(np.float16)).cuda()
    a, b = x.clone(), torch.empty_like(x)
    torch.cuda.synchronize()
    want = single(ctx, x, h, w, layers)
    out = ien.conv3_chain(ctx, a, b, h, w, [m for m, _ in layers], [s for _, s in layers])
    ien.conv3_chain_status(ctx)
    assert same_bits(out, want)
