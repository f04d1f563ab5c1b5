"""The padded PSF correlation on line transforms (csrc/kernels_conv.hip)
against numpy in FP64: every radix and edge of the LDS variants, odd images and
PSFs, images not square, one row or pixel, and an odd padded size (library).

Transforms, product and sums are FP64, so a result differs from numpy's by the
rounding to float, half a unit of 2^-23 of its own size, and some 1e-14 of the
largest: 6.1e-8 and 1e-12 cover both."""
import numpy as np
import pytest

import p9idg

pytestmark = pytest.mark.gpu


def _reference(psf, img):
    """Common.cs:146-160 and PaddedConvolver.cs:50-64."""
    (ph, pw), (H, W) = psf.shape, img.shape
    N0, N1 = H + ph, W + pw
    k = np.zeros((N0, N1))
    y, x = H // 2 + 1, W // 2 + 1
    k[y:y + ph, x:x + pw] = psf[::-1, ::-1]
    h = N0 // 2
    s = k.copy()
    s[:h, :h], s[h:2 * h, h:2 * h] = k[h:2 * h, h:2 * h], k[:h, :h]
    s[:h, h:2 * h], s[h:2 * h, :h] = k[h:2 * h, :h], k[:h, h:2 * h]
    b = np.zeros((N0, N1))
    b[ph // 2:ph // 2 + H, pw // 2:pw // 2 + W] = img
    out = np.fft.irfft2(np.fft.rfft2(s) * np.fft.rfft2(b), s=(N0, N1))
    return out[ph // 2:ph // 2 + H, pw // 2:pw // 2 + W]


@pytest.mark.parametrize("H,W,ph,pw", [
    (8, 8, 8, 8), (1, 3, 5, 3), (13, 13, 1, 1), (15, 15, 3, 3), (62, 60, 18, 20), (63, 63, 31, 31), (64, 64, 15, 15),
    (7, 500, 505, 12), (449, 449, 63, 63), (451, 451, 63, 63), (1000, 1000, 24, 24), (1400, 1400, 58, 58),
    (1900, 1900, 148, 148), (2049, 2049, 101, 101), (3000, 3000, 72, 72), (3001, 3001, 99, 99), (3072, 3072, 192, 192),
    (3700, 3700, 50, 50), (4032, 4032, 64, 64),
])
def test_convolver(H, W, ph, pw):
    rng = np.random.default_rng(H + pw)
    psf = rng.standard_normal((ph, pw)).astype(np.float32)
    ref_img = rng.standard_normal((H, W)).astype(np.float32)
    with p9idg.PaddedConvolver(psf, (H, W)) as conv:
        conv.Convolve(rng.standard_normal((H, W)).astype(np.float32))  # nothing of it stays behind
        out = conv.Convolve(ref_img)
    ref = _reference(psf.astype(np.float64), ref_img.astype(np.float64))
    assert np.all(np.abs(out - ref) <= 6.1e-8 * np.abs(ref) + 1e-12 * np.abs(ref).max())
