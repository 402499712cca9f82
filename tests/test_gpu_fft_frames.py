"""FFT frames of padded canvases, which leave no room beside the canvas for the
kernel: images, likelihoods and gradients against brute force where the canvas
fills its frame exactly, by one pixel more or less, with even and odd kernels,
kernels wider than the image, and (unpadded) a calc region of the image's size."""
import numpy as np
import pytest

import profit_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,kx,ky,padded", [(56, 24, 9, 9, True), (57, 25, 9, 9, True), (55, 23, 9, 9, True),
                                              (50, 40, 15, 25, True), (48, 48, 16, 16, True), (12, 10, 31, 25, True),
                                              (64, 64, 9, 9, False), (237, 220, 41, 41, True)])
def test_frames_do_not_wrap(w, h, kx, ky, padded):
    rng = np.random.default_rng(w * h)
    psf = rng.uniform(0.1, 1.0, (ky, kx))
    # light up to every edge
    comps = [P.make_profile("sersic", convolve=True, xcen=0.5 * w, ycen=0.5 * h, mag=10.0, re=float(max(w, h)), nser=1.0, axrat=0.9),
             P.make_profile("moffat", convolve=True, xcen=1.0, ycen=h - 1.5, mag=9.0, fwhm=4.0, con=3.0)]
    data, sigma = rng.uniform(1e-3, 2e-3, (h, w)), np.full((h, w), 1e-3)
    calc = None if padded else np.ones((h, w), np.uint8)
    got = {}
    for method in ("brute", "fft"):
        eng = P.Engine()
        eng.set_conv_method(method)
        g = eng.add_galaxy(w, h, data, sigma, psf=psf, calcregion=calc, likefunc="norm")
        eng.set_batch([g], [2])
        got[method] = (eng.model_images(comps)[0], *eng.like_grad(comps))
    (ib, lb, gb), (if_, lf, gf) = got["brute"], got["fft"]
    # brute force sums FP32 per kernel column
    assert np.max(np.abs(ib / if_ - 1)) <= 1e-5
    assert np.allclose(lb, lf, rtol=1e-5)
    assert np.all(np.abs(gb - gf).max(axis=0) <= 1e-4 * np.abs(gf).max(axis=0) + 1e-6 * np.abs(gf).max())
