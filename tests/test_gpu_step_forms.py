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


@pytest.mark.parametrize("N,p", [(40_001, 3), (150_001, 3), (150_001, 4)])
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


@pytest.mark.parametrize("D,N,p,small", [(2, 39_999, 3, True), (2, 40_000, 3, False), (2, 39_999, 2, True), (2, 70_000, 3, False),
                                         (2, 40_000, 4, True), (2, 149_999, 5, True), (2, 150_000, 4, False),
                                         (1, 2_000, 3, False)])
def test_which_form_a_step_takes(D, N, p, small):
    """The shared launches only where they were measured to be the faster form, and there the same grid: the step
    equals a batch member's (which always spreads over tables) bit for bit."""
    print(f"[gpu] step forms: D={D} N={N} p={p}", flush=True)
    P, Y = random_csr(N, 6, seed=N), blobs(N, D, 6, seed=p, span=40.0, sd=2.0)
    a = context(P, Y, D, p)
    a.set_timing(True)
    a.step(0.5, 200.0, 5.0)
    names = [str(k) for k in a.kernel_stats()]
    a.set_timing(False)
    assert any("spread_kern" in k for k in names) == small, names
    for _ in range(2):
        a.step(0.5, 200.0, 5.0)
    if D == 2:
        m = context(P, Y, D, p)
        b = fg.Batch([m])
        for _ in range(3):
            b.step([(0.5, 200.0, 5.0)])
        np.testing.assert_array_equal(a.get_Y(), m.get_Y())
        b.close()
        m.close()
    a.close()


@pytest.mark.parametrize("N,p", [(41_000, 3), (150_001, 4)])
def test_spread_workgroup_size_does_not_change_a_2d_step(N, p):
    """Points per workgroup of the table spread, at sizes that take it, host-planned and captured."""
    print(f"[gpu] step forms: spread points N={N} p={p}", flush=True)
    P, Y = random_csr(N, 6, seed=N), blobs(N, 2, 6, seed=p, span=40.0, sd=2.0)
    want = None
    for pts in (1024, 512, 2048, 4096):
        for graph in (False, True):
            c = context(P, Y, 2, p)
            c.set_spread_points(pts)
            g, z = c.gradient()
            if graph:
                c.set_graph(True)
            for _ in range(3):
                c.step(0.5, 200.0, 5.0)
            got = (g, z, c.get_Y())
            c.close()
            want = want or got
            np.testing.assert_array_equal(got[0], want[0])
            assert got[1] == want[1]
            np.testing.assert_array_equal(got[2], want[2])


def test_batch_members_get_their_own_spread_size():
    """Creating a batch tunes every member's table spread, also of those that would not use one alone: 2,000 points
    are two workgroups of 1024 points (the default) or four of 512."""
    sizes = [2000, 2001, 2500]
    print(f"[gpu] step forms: batch tuning {sizes}", flush=True)
    data = [(random_csr(N, 6, seed=N), blobs(N, 2, 4, seed=N, span=30.0, sd=2.0)) for N in sizes]
    single, members = [context(P, Y) for P, Y in data], [context(P, Y) for P, Y in data]
    b = fg.Batch(members)
    assert [c.tuned()[0] for c in members] == [512] * len(sizes)
    for _ in range(3):
        b.step([(0.5, 100.0, 5.0)] * len(sizes))
        for c in single:
            c.step(0.5, 100.0, 5.0)
    for c, m in zip(single, members):
        np.testing.assert_array_equal(c.get_Y(), m.get_Y())
    b.close()
    for c in single + members:
        c.close()
