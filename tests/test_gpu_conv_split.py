"""The brute-force convolution of few tiles (kernel columns in four slices,
tiles in parts) against the one of many and against the FP64 oracle: image
edges inside a tile and inside a part, kernels narrower than the slices or taller
than one LDS chunk, and every tile height."""
import numpy as np
import pytest

import oracle as O
import profit_amd as P
from tests.helpers import gpu_profiles, oracle_profiles, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,kx,ky,rows", [(65, 33, 3, 3, 8), (40, 97, 3, 7, 8), (130, 41, 25, 25, 2), (64, 64, 31, 31, 16),
                                            (63, 85, 9, 71, 4), (183, 70, 31, 31, 8)])
def test_split_equals_whole(w, h, kx, ky, rows):
    rng = np.random.default_rng(kx * ky)
    psf = rng.uniform(0.1, 1.0, (ky, kx))
    comps = [dict(type="moffat", xcen=0.4 * w, ycen=0.6 * h, mag=12.0, fwhm=6.0, con=3.0, ang=30.0, axrat=0.7, box=0.0)]
    spec = O.ModelSpec(w, h, psf=psf, threads=8)
    ref = O.model_evaluate(spec, oracle_profiles(comps))["image"]
    sigma = np.ones((h, w))
    data = 1.1 * ref
    oll, ograd = O.loglike_grad(O.FitSpec(spec, data, sigma, np.ones((h, w), np.uint8), "norm"), oracle_profiles(comps))
    eng = P.Engine()
    eng.set_tile_rows(rows)
    g = eng.add_galaxy(w, h, data, sigma, psf=psf, likefunc="norm")
    images, grads = [], []
    for batch in (1, 700):
        eng.set_batch([g] * batch, [1] * batch)
        params = P.profile_array(gpu_profiles(comps) * batch)
        images.append(eng.model_images(params)[-1])
        ll, grad = eng.like_grad(params)
        assert np.allclose(ll, oll, rtol=1e-9, atol=1e-6)
        grads.append(grad[-1])
        assert rel_err(images[-1], ref)[0] <= 1e-5
        assert np.all(np.abs(grad[-1] - ograd[0]) <= 2e-3 * np.abs(ograd[0]).max())
    # FP64 sums in another order: at most the last FP32 bit of a pixel
    assert np.allclose(images[0], images[1], rtol=1.2e-7, atol=0)
