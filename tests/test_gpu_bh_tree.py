"""The Barnes-Hut tree built on the GPU (and the ordered Z sum) against the oracle's insertions: gradient and Z
equal bit for bit at the edges of the build: the fewest points, chains of one thread (48 points), of one wavefront
(64 to a chunk, 2048 the longest of the second list), the root's chunks (2048), the Z sum's runs (1024 and 16384);
close pairs (deep trees), a far centre, tiny extents, and what goes to the host's insertions (duplicates, pairs
closer than the keys resolve)."""
import time

import numpy as np
import pytest

import fitsne_gpu as fg
import orc

pytestmark = pytest.mark.gpu


def small_P(N, seed):
    rng = np.random.default_rng(seed)
    k = min(3, N - 1)
    row = np.arange(N + 1, dtype=np.uint32) * k
    col = (np.arange(N)[:, None] + 1 + np.arange(k)[None, :]) % N
    val = rng.random(N * k)
    return row, col.reshape(-1).astype(np.uint32), val / val.sum()


def compare(Y, theta, seed=1):
    N, D = Y.shape
    P = small_P(N, seed)
    c = fg.Context(no_dims=D, precision=fg.FP64_BH)
    c.set_theta(theta)
    c.set_P(*P)
    c.set_Y(Y)
    g, z = c.gradient()
    g2, z2 = c.gradient()
    c.close()
    gr, zr = orc.bh_gradient(P, Y, theta)
    np.testing.assert_array_equal(g, gr)
    assert z == zr
    np.testing.assert_array_equal(g2, gr)
    assert z2 == zr


@pytest.mark.parametrize("D", [1, 2, 3])
@pytest.mark.parametrize("N", [2, 3, 5, 47, 48, 49, 50, 64, 65, 129, 1023, 1025, 2047, 2049, 4097])
def test_tree_sizes(N, D):
    rng = np.random.default_rng(N * 10 + D)
    print(f"[gpu] bh tree N={N} D={D}", flush=True)
    compare(rng.normal(0, 5, size=(N, D)), 0.6)


@pytest.mark.parametrize("N,D,theta", [(16385, 2, 0.5), (33000, 2, 0.9), (20000, 3, 0.8), (17000, 1, 0.5)])
def test_tree_clusters(N, D, theta):
    rng = np.random.default_rng(N)
    cen = rng.uniform(-40, 40, size=(20, D))
    Y = cen[rng.integers(0, 20, size=N)] + rng.normal(size=(N, D)) * np.exp(rng.uniform(-6, 1, size=(N, 1)))
    print(f"[gpu] bh tree N={N} D={D} clusters", flush=True)
    compare(Y, theta)


@pytest.mark.parametrize("name", ["close_pairs", "closer_pairs", "close_group", "too_close", "duplicates", "far", "tiny", "line", "one_far", "lattice"])
@pytest.mark.parametrize("D", [1, 2, 3])
def test_tree_awkward(name, D):
    rng = np.random.default_rng(7)
    N = 3000
    Y = rng.normal(0, 3, size=(N, D))
    if name == "close_pairs":
        Y[1000:1400] = Y[:400] + 1e-5 * rng.normal(size=(400, D))
    elif name == "closer_pairs":  # equal first keys in 2D and 3D
        Y[1000:1400] = Y[:400] + 1e-11 * rng.normal(size=(400, D))
    elif name == "close_group":  # runs of equal first keys, one longer than a thread sorts
        Y[1000:1040] = Y[0] + 1e-12 * rng.normal(size=(40, D))
        if D == 2:
            Y[1100:1200] = Y[1] + 1e-12 * rng.normal(size=(100, D))
    elif name == "too_close":
        Y[1000:1010] = Y[:10] * (1 + 4e-16)
    elif name == "duplicates":
        Y[1000:1400] = Y[:400]
        Y[2000] = Y[0]
    elif name == "far":
        Y += 1e7
    elif name == "tiny":
        Y *= 1e-9
    elif name == "line":
        Y[:, 0] = np.linspace(-1, 1, N)
        Y[:, 1:] = 0.25
    elif name == "one_far":
        Y[17] = 1e5
    else:
        Y = rng.permutation(np.arange(N))[:, None] // np.array([1, 60, 600])[None, :D] % 50 - 25.0
        Y = np.unique(Y, axis=0)
        Y = Y[rng.permutation(len(Y))]
    print(f"[gpu] bh tree {name} D={D}", flush=True)
    compare(np.ascontiguousarray(Y), 0.5)


@pytest.mark.parametrize("scale", [1.0, 1e-3])
def test_steps_follow_the_host_loop(scale):
    """20 steps with the tree rebuilt each time stay with the oracle's loop."""
    N, D = 5000, 2
    rng = np.random.default_rng(3)
    Y = rng.normal(0, 4, size=(N, D)) * scale
    P = small_P(N, 4)
    c = fg.Context(no_dims=D, precision=fg.FP64_BH)
    c.set_P(*P)
    c.set_Y(Y)
    for _ in range(20):
        c.step(0.8, 200.0)
        Yg = c.get_Y()
        g, z = c.gradient()
        gr, zr = orc.bh_gradient(P, Yg, 0.5)
        np.testing.assert_array_equal(g, gr)
        assert z == zr
    c.close()


@pytest.mark.parametrize("scale", [1e126, 1e128, 1e160])
@pytest.mark.parametrize("N", [17, 1100])
def test_far_apart(N, scale):
    """Q so small that Z lies below the range the parallel sum folds, or is zero (then dC is not a number)."""
    rng = np.random.default_rng(N)
    print(f"[gpu] bh far apart N={N} scale={scale}", flush=True)
    with np.errstate(all="ignore"):
        compare(rng.normal(size=(N, 2)) * scale, 0.5)


@pytest.mark.parametrize("D", [2, 3])
def test_overlap_off(D):
    """One kernel after another: the same bits, and kernel times that add up to no more than the call."""
    N = 60_000
    print(f"[gpu] bh overlap off D={D}", flush=True)
    Y = np.random.default_rng(D).normal(size=(N, D)) * 20
    P, out = small_P(N, 1), []
    for overlap in (True, False):
        c = fg.Context(no_dims=D, precision=fg.FP64_BH)
        c.set_overlap(overlap)
        c.set_P(*P)
        c.set_Y(Y)
        c.gradient()
        c.set_timing(True)
        t = time.perf_counter()
        g, z = c.gradient()
        t = (time.perf_counter() - t) * 1e3
        if not overlap:
            ms = sum(m for _, m in c.kernel_stats().values())
            assert ms <= t, (ms, t)
        out.append((g, z))
        c.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]


@pytest.mark.parametrize("N,D", [(699, 1), (699, 2), (700, 1), (700, 2), (701, 2), (255, 3), (256, 3), (257, 3)])
def test_about_the_host_line(N, D):
    print(f"[gpu] bh host line N={N} D={D}", flush=True)
    compare(np.random.default_rng(N + D).normal(0, 5, size=(N, D)), 0.6)


def test_builds_that_end_on_the_host():
    """Coinciding points send this and the next trees to the host; a new Y starts anew, between calls of both kinds."""
    N = 2000
    print("[gpu] bh host builds", flush=True)
    rng = np.random.default_rng(9)
    Y = rng.normal(0, 5, size=(N, 2))
    Yd = Y.copy()
    Yd[100:300] = Yd[:200]
    P = small_P(N, 2)
    c = fg.Context(no_dims=2, precision=fg.FP64_BH)
    c.set_P(*P)
    for V, calls in ((Yd, 7), (Y, 3), (Yd, 2), (Y, 1)):
        c.set_Y(V)
        gr, zr = orc.bh_gradient(P, V, 0.5)
        for _ in range(calls):
            g, z = c.gradient()
            np.testing.assert_array_equal(g, gr)
            assert z == zr
    c.set_Y(Yd)
    for _ in range(24):  # the pairs part after the first step; the GPU's trees come back on their own
        c.step(0.5, 100.0)
    V = c.get_Y()
    g, z = c.gradient()
    gr, zr = orc.bh_gradient(P, V, 0.5)
    np.testing.assert_array_equal(g, gr)
    assert z == zr
    c.close()
