"""GPU: the spectral branch's launches on maps with a side of 65 .. 128, each
transform against float64 on the operands that the launch reads.

These maps' transforms are products in f32 (ien_fourier's passes on f32 MFMA),
computed here on f16 and bf16 matrix cores from split operands.  Each must be
no further from float64 than ien_fourier's pass on the same operand: in 2-norm
where f32 comes out, and where f16 comes out by the share of values that are
not the float64 result rounded once, which grows with the error (three
standard deviations of the difference of two such counts allowed).  Operands
held in two halves of f16 miss that four times over, without their lower
halves by hundreds."""

import numpy as np
import pytest

import synthetic
from internal import LongSpectral

pytestmark = pytest.mark.gpu

LOCAL, GLOBAL, CHANNELS, SPECTRAL = 128, 384, 512, 192
# Either side over 64 and both; the smallest and largest of each, odd and even
# ones, lines that end within a block of 16 and 32.
SHAPES = [(65, 128), (128, 65), (128, 128), (125, 85), (2, 65), (65, 2), (1, 100), (100, 1), (40, 127), (97, 33)]


@pytest.fixture(scope="module")
def weights():
    t = synthetic.lama_tensors()
    return {k: t[f"block3.ffc0.{k}"] for k in ("spectral_in.weight", "spectral_in.bias")}


def dft(n):
    a = 2 * np.pi * (np.outer(np.arange(n), np.arange(n)) % n) / n
    return np.cos(a), np.sin(a)


def off32(got, want):
    return np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-300)


def off16(got, want):
    """The number of values of got (f16) that are not want rounded once."""
    return int(np.sum(got != want.astype(np.float16)))


def no_further(what, new, old, counts=False):
    print(f"  {what}: {new:.4g} here, {old:.4g} in the f32 passes", flush=True)
    assert new <= old + (3 * np.sqrt(new + old) if counts else 1e-9), (what, new, old)  # (1e-9: lines of one or two)


@pytest.mark.parametrize("h,w", SHAPES)
def test_transforms_keep_f32_accuracy(ctx, weights, h, w):
    import torch
    import ien

    print(f"long spectral {h}x{w}", flush=True)
    half, rng = w // 2 + 1, np.random.default_rng(h * 1000 + w)
    kyb = (h + 31) // 32
    sp = LongSpectral(ctx, h, w)
    m_in = ien.Matrix(ctx, weights["spectral_in.weight"], weights["spectral_in.bias"])
    m_f = ien.Matrix(ctx, np.eye(2 * SPECTRAL, dtype=np.float32), np.zeros(2 * SPECTRAL, np.float32))
    m_out = ien.Matrix(ctx, np.concatenate([np.eye(SPECTRAL), -np.eye(SPECTRAL)], 1).astype(np.float32))
    x = torch.from_numpy(rng.standard_normal((h, w, CHANNELS)).astype(np.float16)).cuda()
    spectral = torch.empty((h, SPECTRAL, w), dtype=torch.float16, device="cuda")
    r = torch.empty((h, w, SPECTRAL), dtype=torch.float32, device="cuda")
    z = torch.empty(half * kyb * 32 * 2 * SPECTRAL, dtype=torch.float16, device="cuda")
    u = torch.empty((h, half, 2 * SPECTRAL), dtype=torch.float32, device="cuda")
    out = torch.zeros((h, w, GLOBAL), dtype=torch.float16, device="cuda")
    flat = torch.zeros_like(spectral)
    torch.cuda.synchronize()  # (the library's stream need not be torch's)
    sp.rows(x[..., LOCAL:], CHANNELS, m_in, spectral, r)
    sp.columns(m_f, r, z, u)
    sp.back(m_out, flat, u, out, GLOBAL)
    # The f32 passes, each on the operand that the launch above read.
    f = ien.Fourier(ctx, h, w)
    torch.cuda.synchronize()
    rows = spectral.transpose(1, 2).contiguous()
    work = torch.empty((h, half, 2 * SPECTRAL), dtype=torch.float32, device="cuda")
    spectrum = torch.empty((h, half, 2 * SPECTRAL), dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    f.forward(rows, SPECTRAL, SPECTRAL, work, spectrum)
    # z is the product's operand: [column][block of 32 rows][16 channels][half][row][8].
    zp = z.view(half, kyb, 2 * SPECTRAL // 16, 2, 32, 8).permute(0, 1, 4, 2, 3, 5)
    zp = zp.reshape(half, kyb * 32, 2 * SPECTRAL)[:, :h]
    filtered = zp.permute(1, 0, 2).clamp(min=0).contiguous()  # (the fourier matrix is the identity)
    work2, added = torch.empty_like(work), torch.zeros((h, w, SPECTRAL), dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    f.inverse(filtered, SPECTRAL, work2, added, SPECTRAL)
    torch.cuda.synchronize()
    s = spectral.double().cpu().numpy().transpose(0, 2, 1)  # [y][x][c]
    r, u, work, work2 = (t.double().cpu().numpy() for t in (r, u, work, work2))
    zp, spectrum, filtered, out, added = (t.cpu().numpy() for t in (zp, spectrum, filtered, out, added))
    scale = 1.0 / np.sqrt(h * w)
    cw, sw = dft(w)
    ch, sh = dft(h)

    # Row transform: real parts of columns 0 .. w / 2, then the imaginary
    # parts of columns 1 ..  (R as [y][k][re | im], as ien_fourier's.)
    want = np.concatenate([np.einsum("kx,yxc->ykc", cw[:half], s), np.einsum("kx,yxc->ykc", -sw[:half], s)], -1)
    full = np.zeros_like(want)
    full[..., :SPECTRAL] = r[:, :half]
    full[:, 1:w - half + 1, SPECTRAL:] = r[:, half:]
    no_further("rows", off32(full, want), off32(work, want))

    def columns(a):  # of [y][k][re | im], to [ky][k][re | im]
        re, im = a[..., :SPECTRAL], a[..., SPECTRAL:]
        return scale * np.concatenate([np.einsum("ky,ymc->kmc", ch, re) + np.einsum("ky,ymc->kmc", sh, im),
                                       np.einsum("ky,ymc->kmc", ch, im) - np.einsum("ky,ymc->kmc", sh, re)], -1)

    no_further("columns", off16(zp.transpose(1, 0, 2), columns(full)), off16(spectrum, columns(work)), True)

    # Inverse columns.
    p = filtered.astype(np.float64)
    pr, pi = p[..., :SPECTRAL], p[..., SPECTRAL:]
    want = np.concatenate([np.einsum("ky,kmc->ymc", ch, pr) - np.einsum("ky,kmc->ymc", sh, pi),
                           np.einsum("ky,kmc->ymc", sh, pr) + np.einsum("ky,kmc->ymc", ch, pi)], -1)
    no_further("inverse columns", off32(u, want), off32(work2, want))

    # Inverse rows onto a map of zeros.
    edge = (np.arange(half) == 0) | (2 * np.arange(half) == w)
    wk = np.where(edge, 1.0, 2.0)[:, None]
    imag = np.where(edge[:, None], 0.0, -wk * sw[:half])

    def inverse_rows(a):
        return scale * (np.einsum("kx,ykc->yxc", wk * cw[:half], a[..., :SPECTRAL]) +
                        np.einsum("kx,ykc->yxc", imag, a[..., SPECTRAL:]))

    got = np.where(out[..., :SPECTRAL] > 0, out[..., :SPECTRAL], -out[..., SPECTRAL:])
    no_further("inverse rows", off16(got, inverse_rows(u)), off16(added, inverse_rows(work2)), True)
    f.free()
    for m in (sp, m_in, m_f, m_out):
        m.free()


def test_back_adds_to_the_map_in_place(ctx):
    """The wide back launch with a cross output to accumulate onto, a strided
    map and a residual, against float64."""
    import torch
    import ien

    h, w = 66, 90
    half, rng = w // 2 + 1, np.random.default_rng(5)
    sp = LongSpectral(ctx, h, w)
    wt = (rng.standard_normal((SPECTRAL, GLOBAL)) / 16).astype(np.float32)
    m_out = ien.Matrix(ctx, wt)
    s = rng.standard_normal((h, w, SPECTRAL)).astype(np.float16)
    cross = rng.standard_normal((h, w, CHANNELS)).astype(np.float16)
    add = rng.standard_normal((h, w, CHANNELS)).astype(np.float16)
    d_s = torch.from_numpy(np.ascontiguousarray(s.transpose(0, 2, 1))).cuda()
    u = torch.zeros((h, half, 2 * SPECTRAL), dtype=torch.float32, device="cuda")
    d_out, d_add = torch.from_numpy(cross).cuda(), torch.from_numpy(add).cuda()
    torch.cuda.synchronize()
    sp.back(m_out, d_s, u, d_out[..., LOCAL:], CHANNELS, d_add[..., LOCAL:], d_add[..., LOCAL:])
    torch.cuda.synchronize()
    got = d_add.cpu().numpy()
    assert np.array_equal(got[..., :LOCAL], add[..., :LOCAL])
    assert np.array_equal(d_out.cpu().numpy(), cross)
    w16 = wt.astype(np.float16).astype(np.float64)
    acc = cross[..., LOCAL:].astype(np.float64) + s.astype(np.float64) @ w16
    want = np.maximum(acc, 0).astype(np.float16).astype(np.float64) + add[..., LOCAL:]
    # Two roundings to f16, each within half a spacing of up to 2^-10 of a
    # value (which sums in f32 may move over a boundary: one spacing more).
    spacing = 2.0 ** -10 * np.maximum(np.abs(want), np.maximum(np.abs(acc), 2.0 ** -14))
    assert np.all(np.abs(got[..., LOCAL:] - want) <= 2 * spacing)
    for m in (sp, m_out):
        m.free()
