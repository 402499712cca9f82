"""Invalid parameters in a batch: the component whose set-up fails draws nothing
(on the CPU, tests/native/setup_error.cpp), every evaluation entry point reports
the error, and the engine's next evaluation is right."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_failed_setup_leaves_an_undrawn_component(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "setup_error")
    r = subprocess.run([gxx, "-std=c++20", "-O1", "-w", "-ffp-contract=off", "-pthread",
                        "-I" + os.path.join(ROOT, "tests", "native", "hip_cpu"), "-I" + os.path.join(ROOT, "profit_amd", "csrc"),
                        os.path.join(ROOT, "tests", "native", "setup_error.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.count("ok ") == 9, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("bad,message", [(dict(axrat=0.0), "axrat"), (dict(nser=-1.0), "nser"), (dict(max_recursions=31), "max_recursions"),
                                         (dict(adjust=False, resolution=100), "resolution")])
def test_errors_are_reported_and_leave_the_engine_usable(bad, message):
    import profit_amd as P
    w, h = 60, 50
    par = dict(xcen=30.2, ycen=24.7, mag=15.0, re=5.0, nser=2.0, ang=30.0, axrat=0.6)
    good = [P.make_profile("sersic", **par), P.make_profile("moffat", xcen=20.0, ycen=20.0, mag=16.0, fwhm=3.0, con=2.5)]
    wrong = [P.make_profile("sersic", **dict(par, **bad)), good[1]]

    def engine():
        eng = P.Engine()
        eng.set_batch([eng.add_galaxy(w, h, np.zeros((h, w)), np.ones((h, w)), likefunc="norm", magzero=30.0)], [2])
        return eng

    ref = engine()
    image, (ll, grad) = ref.model_images(good)[0], ref.like_grad(good)
    eng = engine()
    for call in (eng.like, eng.like_grad, eng.model_images, eng.diagnostics):
        with pytest.raises(Exception, match=message):
            call(wrong)
        assert np.array_equal(eng.model_images(good)[0], image)
        got = eng.like_grad(good)
        assert np.allclose(got[0], ll, rtol=1e-12) and np.allclose(got[1], grad, rtol=1e-6, atol=1e-9 * np.abs(grad).max())
