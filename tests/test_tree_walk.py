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


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 5])
def test_overflowing_trees_are_walked_again(n):
    """An n = 8 cusp at acc = 0.01 refines every cell within some 60 cells of
    the centre on each of 6 levels, the last cells of its pixel: more pending nodes than the stack holds.
    The evaluation runs again with the mask walk and equals the oracle."""
    import oracle as O
    import profit_amd as P
    w = h = 8
    par = dict(xcen=4.99999, ycen=3.99999, mag=10.0, re=3.0, nser=8.0, ang=20.0, axrat=0.8, adjust=False, acc=0.01,
               rscale_switch=0.7, rscale_max=50.0, resolution=16, max_recursions=5)
    ref = O.model_evaluate(O.ModelSpec(w, h, threads=8), [O.make_profile("sersic", **par)])["image"]
    eng = P.Engine()
    g = eng.add_galaxy(w, h, np.zeros((h, w)), np.ones((h, w)), likefunc="norm")
    eng.set_batch([g] * n, [1] * n)
    for img in eng.model_images([P.make_profile("sersic", **par)] * n):
        assert np.max(np.abs(img - ref) / ref) <= 1e-5
    ll = eng.like([P.make_profile("sersic", **par)] * n)
    assert np.allclose(ll, -0.5 * np.sum(ref ** 2) - 0.5 * w * h * np.log(2 * np.pi), rtol=2e-5)
