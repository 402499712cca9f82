"""The tree walk of the sub-sampled pixels on the CPU (tests/native/tree_walk.cpp):
one host thread per GPU thread under AddressSanitizer, against a plain
recursion, and an evaluation whose trees overflow the walk's stack on the GPU."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "profit_amd", "csrc")


def test_tree_walk_equals_the_recursion(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "tree_walk")
    r = subprocess.run([gxx, "-std=c++20", "-O1", "-g", "-w", "-ffp-contract=off", "-fsanitize=address", "-pthread",
                        "-I" + os.path.join(ROOT, "tests", "native", "hip_cpu"), "-I" + CSRC,
                        os.path.join(ROOT, "tests", "native", "tree_walk.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300, env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, r.stdout + r.stderr[-4000:]
    assert r.stdout.count("ok ") == 16, r.stdout


def test_sub_pixel_kernels_equal_the_recursion(tmp_path):
    """The kernels around the walk (tests/native/tree_kernels.cpp), with a stack of
    64 nodes a wavefront so that small trees overflow it."""
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    header = open(os.path.join(CSRC, "kernel_common.h")).read()
    assert "constexpr int kTreeShare = 256;" in header
    (tmp_path / "kernel_common.h").write_text(header.replace("constexpr int kTreeShare = 256;", "constexpr int kTreeShare = 64;"))
    exe = str(tmp_path / "tree_kernels")
    r = subprocess.run([gxx, "-std=c++20", "-O1", "-g", "-w", "-ffp-contract=off", "-fsanitize=address", "-pthread",
                        "-I" + os.path.join(ROOT, "tests", "native", "hip_cpu"), "-I" + str(tmp_path), "-I" + CSRC,
                        os.path.join(ROOT, "tests", "native", "tree_kernels.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600, env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0 and r.stdout.count("ok ") == 6, r.stdout + r.stderr[-4000:]


# one component whose tree overflows the stack of a block of twelve wavefronts and
# one whose tree overflows that of a block of four (walked so among many components)
CUSP = dict(mag=-2.0, adjust=False, resolution=16, rscale_max=50.0)
OVERFLOWS = [("coresersic", 1, dict(CUSP, xcen=1 - 3.3e-10, ycen=1 - 3.3e-10, ang=45.0, axrat=0.3, re=6.0, rb=2.0, nser=3.0, a=2.0,
                                    b=1.7, acc=0.1, rscale_switch=0.4, max_recursions=10)),
             ("sersic", 1100, dict(CUSP, xcen=5 - 1e-5, ycen=4 - 1e-5, ang=20.0, axrat=0.8, re=3.0, nser=8.0, acc=0.05,
                                   rscale_switch=0.3, max_recursions=5))]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,par", OVERFLOWS)
def test_overflowing_trees_are_walked_by_masks(kind, n, par):
    """The first evaluation with a tree that overflows the walk's stack runs again
    with the mask walk behind the tree walk; later ones run once (from the graph
    where there is one) and all equal the oracle."""
    import oracle as O
    import profit_amd as P
    w = h = 8
    op = [O.make_profile(kind, **par)]
    ref = O.model_evaluate(O.ModelSpec(w, h, threads=8), op)["image"]
    sigma = np.full((h, w), 0.1 * ref.mean())
    data = ref + sigma * np.random.default_rng(5).standard_normal((h, w))
    gp = [P.make_profile(kind, **par)]
    # the other components make the family too large for blocks of twelve wavefronts
    plain = [P.make_profile(kind, xcen=4.0, ycen=4.0, mag=20.0, re=2.0, nser=1.0, rough=True)] * (n - 1)
    eng = P.Engine()
    g = eng.add_galaxy(w, h, data, sigma, likefunc="norm")
    eng.set_batch([g, g] if plain else [g], [1, n - 1] if plain else [1])
    params = P.profile_array(gp + plain)
    fit = O.FitSpec(O.ModelSpec(w, h, threads=8), data, sigma, np.ones((h, w), np.uint8), "norm")
    oll = O.loglike(fit, op)
    for k in range(3):
        img = eng.model_images(params)[0]
        assert eng.walk_stats()["overflowed"] > 0
        assert np.max(np.abs(img - ref) / ref) <= 1e-5
        # FP32 pixels: 1e-5 of each against sigma = 0.1 of the mean
        ll = eng.like(params)
        assert abs(ll[0] - oll) <= 1e-3 + 1e-6 * abs(oll)
        ll2, grad = eng.like_grad(params)
        assert eng.walk_stats()["overflowed"] > 0
        assert abs(ll2[0] - oll) <= 1e-3 + 1e-6 * abs(oll)
        assert np.all(np.isfinite(grad))
        if k:
            assert np.allclose(grad[0], first, rtol=1e-5, atol=1e-6 * np.abs(first).max())
        first = grad[0]
        assert eng.walk_stats()["repeats"] == 1
    if kind == "sersic":
        og = O.loglike_grad(fit, op)[1][0]
        assert np.all(np.abs(grad[0] - og)[:9] <= 2e-3 * np.maximum(np.abs(og), 5e-2 * np.abs(og).max())[:9])
    # a new batch starts without the mask walk
    eng.set_batch([g], [1])
    eng.like([P.make_profile(kind, xcen=4.0, ycen=4.0, mag=0.0, re=2.0, nser=1.0)])
    assert eng.walk_stats() == {"overflowed": 0, "repeats": 1}
