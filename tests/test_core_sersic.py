"""Core-Sersic profiles of sharp transitions (shape parameter a), whose powers
r^a leave FP32's range: the FP32 forms on the CPU (tests/native/core_sersic.cpp)
and images, likelihoods and gradients on the GPU against the FP64 oracle."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_fp32_forms_equal_fp64(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "core_sersic")
    r = subprocess.run([gxx, "-std=c++20", "-O2", "-w", "-ffp-contract=off", "-pthread",
                        "-I" + os.path.join(ROOT, "tests", "native", "hip_cpu"), "-I" + os.path.join(ROOT, "profit_amd", "csrc"),
                        os.path.join(ROOT, "tests", "native", "core_sersic.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok "), r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("a,rb", [(2.0, 3.0), (12.0, 20.0), (25.0, 3.0), (40.0, 14.0)])
def test_sharp_transitions(a, rb):
    import oracle as O
    import profit_amd as P
    w, h = 90, 70
    par = dict(xcen=45.001, ycen=35.499, mag=14.0, ang=30.0, axrat=0.7, re=33.0, rb=rb, nser=2.0, a=a, b=0.6)
    spec = O.ModelSpec(w, h, magzero=30.0, threads=8)
    op = [O.make_profile("coresersic", **par)]
    ref = O.model_evaluate(spec, op)["image"]
    sigma = np.sqrt(np.abs(ref) + 1.0)
    data = 1.05 * ref + sigma * np.random.default_rng(3).standard_normal((h, w))
    eng = P.Engine()
    eng.set_batch([eng.add_galaxy(w, h, data, sigma, likefunc="norm", magzero=30.0)], [1])
    gp = [P.make_profile("coresersic", **par)]
    img = eng.model_images(gp)[0]
    assert np.max(np.abs(img - ref) / ref) <= 1e-5
    ll, grad = eng.like_grad(gp)
    fit = O.FitSpec(spec, data, sigma, np.ones((h, w), np.uint8), "norm")
    assert np.allclose(ll, O.loglike(fit, op), rtol=1e-6)
    # the oracle's gradient of a core-Sersic is by differences: steps and gate of the batch test
    steps = np.full((1, O.NGRAD), 1e-6)
    steps[:, :2] = 1e-8
    o = O.loglike_grad_fd(fit, op, rel_step=steps)[1][0]
    slots = [0, 1, 2, 3, 4, 6, 7, 8, 9, 10]
    print(f"[core] a {a}: gpu {np.array2string(grad[0], precision=4)} fd {np.array2string(o, precision=4)}", flush=True)
    assert np.all(np.abs(grad[0] - o)[slots] <= 2e-3 * np.maximum(np.abs(o), 5e-2 * np.abs(o[slots]).max())[slots])
