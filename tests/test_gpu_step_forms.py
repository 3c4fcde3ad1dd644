"""The forms of a host-planned FP32 2D step (passes that share launches on one stream, or the attractive term and the
kernel spectra on a second stream) at sizes that take them: each gives, bit for bit, what the kernels give one
after another."""
import numpy as np
import pytest

import fitsne_gpu as fg
from datagen import blobs, random_csr

pytestmark = pytest.mark.gpu


def context(P, Y, D=2, p=3):
    c = fg.Context(no_dims=D, precision=fg.FP32, n_interpolation_points=p)
    c.set_P(*P)
    c.set_Y(Y)
    return c


@pytest.mark.parametrize("N,p", [(150_001, 3), (150_001, 4)])
def test_streams_leave_results_bitwise_unchanged(N, p):
    """Overlap on and off, across a wider Y (a longer FFT line, so that the spectra's buffers grow) and back."""
    print(f"[gpu] step forms: overlap N={N} p={p}", flush=True)
    P, Y = random_csr(N, 6, seed=N), blobs(N, 2, 8, seed=N, span=25.0, sd=2.0)
    a, b = context(P, Y, p=p), context(P, Y, p=p)
    b.set_overlap(False)
    lens = []
    for Yp in (None, 3.0 * Y, Y):
        if Yp is not None:
            a.set_Y(Yp)
            b.set_Y(Yp)
        for k in range(4):
            za = a.step(0.5, 200.0, 5.0, want_sumq=(k == 3))
            zb = b.step(0.5, 200.0, 5.0, want_sumq=(k == 3))
            assert za == zb
        lens.append(a.last_geometry()["fft_len"])
        np.testing.assert_array_equal(a.get_Y(), b.get_Y())
    assert lens[1] > lens[0]
    ga, za = a.gradient()
    gb, zb = b.gradient()
    np.testing.assert_array_equal(ga, gb)
    assert za == zb
    a.close()
    b.close()
