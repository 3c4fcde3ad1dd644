"""The spread by wavefronts straight into the grid (below 150,000 points) against the oracle, at the edges of the 128
points of a wavefront, with more boxes than points, all but two points in one box, 2 to 5 nodes per box, and on both
sides of the line, where the grid must not depend on the form: a context of N points against the same points
stepped as a batch, and the step repeated, bit for bit."""
import numpy as np
import pytest

import fitsne_gpu as fg
import orc
from datagen import blobs, random_csr

pytestmark = pytest.mark.gpu
TOL = 1e-4  # the FP32 form's bound


def gradient(Y, P, D, df=1.0, p=3):
    c = fg.Context(no_dims=D, precision=fg.FP32, df=df, n_interpolation_points=p)
    c.set_P(*P)
    c.set_Y(Y)
    g, z = c.gradient()
    g2, z2 = c.gradient()
    c.close()
    np.testing.assert_array_equal(g, g2)
    assert z == z2
    return g, z


def compare(Y, D, df=1.0, p=3):
    P = random_csr(len(Y), 6, seed=len(Y))
    Y = Y.astype(np.float32).astype(np.float64)
    g, z = gradient(Y, P, D, df, p)
    want, zw = orc.gradient(P, Y, p=p, df=df)
    r = np.linalg.norm(g - want) / np.linalg.norm(want)
    print(f"    rel={r:.2e}", flush=True)
    assert r <= TOL and abs(z - zw) <= TOL * abs(zw)


@pytest.mark.parametrize("D", [1, 2])
@pytest.mark.parametrize("N", [7, 127, 128, 129, 255, 257, 2047, 2049])
def test_edges(N, D):
    print(f"[gpu] spread wave N={N} D={D}", flush=True)
    compare(blobs(N, D, 4, seed=N, span=30.0, sd=2.0), D)


@pytest.mark.parametrize("D", [1, 2])
@pytest.mark.parametrize("p", [2, 3, 4, 5])
def test_nodes_per_box(p, D):
    print(f"[gpu] spread wave p={p} D={D}", flush=True)
    compare(blobs(3001, D, 5, seed=p, span=30.0, sd=2.0), D, p=p)


@pytest.mark.parametrize("D", [1, 2])
def test_one_box(D):
    print(f"[gpu] spread wave one box D={D}", flush=True)
    rng = np.random.default_rng(D)
    Y = rng.uniform(1.05, 1.35, size=(1000, D))
    Y[0], Y[1] = 25.0, -25.0
    compare(Y, D)


@pytest.mark.parametrize("N", [149999, 150000])
def test_both_sides_of_the_line(N):
    print(f"[gpu] spread wave line N={N}", flush=True)
    compare(blobs(N, 2, 12, seed=N, span=50.0, sd=2.0), 2)


@pytest.mark.parametrize("p", [3, 4])
def test_batch_equals_single(p):
    print(f"[gpu] spread wave batch p={p}", flush=True)
    sizes = [130, 2500, 9001]
    single, members = [], []
    for k in range(2):
        for N in sizes:
            c = fg.Context(no_dims=2, precision=fg.FP32, n_interpolation_points=p)
            c.set_P(*random_csr(N, 6, seed=N))
            c.set_Y(blobs(N, 2, 4, seed=N, span=30.0, sd=2.0))
            (single if k == 0 else members).append(c)
    for c in single:
        for _ in range(3):
            c.step(0.5, 100.0, 5.0)
    b = fg.Batch(members)
    for _ in range(3):
        b.step((0.5, 100.0, 5.0))
    for a, m in zip(single, members):
        np.testing.assert_array_equal(a.get_Y(), m.get_Y())
    b.close()
    for c in single + members:
        c.close()
