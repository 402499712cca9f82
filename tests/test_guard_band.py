"""The guard band of the FP32 refinement test: the FP32 test against the FP64 one
on the CPU over all families' parameters (tests/native/guard_band.cpp), and trees
on the GPU, bit-exact, where the shape parameters amplify FP32 errors."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_fp32_leaves_undecided_cells_to_fp64(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "guard_band")
    r = subprocess.run([gxx, "-std=c++20", "-O2", "-w", "-ffp-contract=off", "-pthread",
                        "-I" + os.path.join(ROOT, "tests", "native", "hip_cpu"), "-I" + os.path.join(ROOT, "profit_amd", "csrc"),
                        os.path.join(ROOT, "tests", "native", "guard_band.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe, "1000"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.count("ok ") == 6, r.stdout


EDGE = dict(adjust=False, rscale_switch=1.1, rscale_max=1.5, resolution=10, max_recursions=2, acc=0.03, box=0.0, mag=15.0)
AMPLIFIED = [
    dict(type="king", xcen=40.3, ycen=39.6, ang=30.0, axrat=0.7, rc=2.5, rt=17.0, a=8.0),
    dict(type="king", xcen=40.5, ycen=40.5, ang=70.0, axrat=0.9, rc=9.0, rt=14.0, a=9.7),
    dict(type="ferrer", xcen=40.2, ycen=39.9, ang=10.0, axrat=0.8, rout=14.0, a=1.0, b=1.95),
    dict(type="ferrer", xcen=40.2, ycen=39.9, ang=10.0, axrat=0.8, rout=14.0, a=5.0, b=1.99),
    dict(type="moffat", xcen=40.1, ycen=40.4, ang=55.0, axrat=0.3, fwhm=9.0, con=900.0),
    dict(type="sersic", xcen=40.5, ycen=40.0, ang=55.0, axrat=0.1, re=9.0, nser=0.25),
    dict(type="coresersic", xcen=40.2, ycen=40.3, ang=20.0, axrat=0.6, re=9.0, rb=4.0, nser=2.0, a=30.0, b=0.8),
]


@pytest.mark.gpu
@pytest.mark.parametrize("k", range(len(AMPLIFIED)))
def test_trees_bit_exact(k):
    import oracle as O
    import profit_amd as P
    from tests.helpers import gpu_profiles, oracle_profiles
    comps = [dict(AMPLIFIED[k], **EDGE)]
    w = h = 80
    ref = O.model_evaluate(O.ModelSpec(w, h, threads=8), oracle_profiles(comps, convolve=False), diag=True)
    eng = P.Engine()
    eng.set_batch([eng.add_galaxy(w, h, np.zeros((h, w)), np.ones((h, w)))], [1])
    cls, nodes = eng.diagnostics(gpu_profiles(comps, convolve=False))
    print(f"[band] {comps[0]['type']}: nodes {int(np.sum(ref['nodes']))}", flush=True)
    assert np.array_equal(cls, ref["cls"].astype(np.int32))
    assert np.array_equal(nodes, ref["nodes"].astype(np.int32))
