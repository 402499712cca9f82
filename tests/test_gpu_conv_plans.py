"""Repeated bare convolutions of one geometry: the kept device set-up must not
let one call's inputs reach another (source, kernel, mask given and then not),
from several threads at once, after its release, and against a direct sum."""
import threading

import numpy as np
import pytest

import profit_amd as P

pytestmark = pytest.mark.gpu


def _inputs(seed, w, h, kw, kh):
    g = np.random.default_rng(seed)
    return g.standard_normal((h, w)), g.uniform(0.1, 1.0, (kh, kw)), (g.uniform(size=(h, w)) < 0.7).astype(np.uint8)


def _direct(src, krn, mask):
    h, w = src.shape
    kh, kw = krn.shape
    pad = np.zeros((h + 2 * kh, w + 2 * kw))
    pad[kh:kh + h, kw:kw + w] = src
    out = np.zeros((h, w))
    for y in range(kh):
        for x in range(kw):
            # the centre tap of an even kernel is K - 1 - K / 2
            oy, ox = kh + (kh - 1 - kh // 2) - y, kw + (kw - 1 - kw // 2) - x
            out += krn[y, x] * pad[oy:oy + h, ox:ox + w]
    return out if mask is None else out * mask


@pytest.mark.parametrize("convolver", ["brute", "fft"])
@pytest.mark.parametrize("w,h,kw,kh", [(40, 31, 5, 9), (130, 70, 25, 25), (64, 64, 64, 64), (9, 9, 1, 1)])
def test_repeated_calls(convolver, w, h, kw, kh):
    sets = [_inputs(s, w, h, kw, kh) for s in range(3)]
    for k in (0, 1, 2, 0):
        src, krn, mask = sets[k]
        for m in (None, mask, None):
            ref = _direct(src, krn, m)
            got = P.convolve(src, krn, mask=m, convolver=convolver)
            # FP32 source and result, FP32 sums per kernel column (brute)
            assert np.max(np.abs(got - ref)) <= 3e-6 * np.abs(krn).sum() * np.abs(src).max()
        P.clear_cache()


def test_threads_do_not_share_a_plan():
    shapes = [(60, 50, 7, 7), (60, 50, 7, 7), (33, 90, 11, 5), (120, 20, 9, 9)]
    refs, errors = {}, []
    for k, s in enumerate(shapes):
        src, krn, mask = _inputs(k, *s)
        refs[k] = (src, krn, mask, P.convolve(src, krn, mask=mask, convolver="fft"))

    def work(k):
        src, krn, mask, ref = refs[k % len(shapes)]
        for _ in range(20):
            if not np.array_equal(P.convolve(src, krn, mask=mask, convolver="fft"), ref):
                errors.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
