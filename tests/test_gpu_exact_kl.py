"""The exact path's KL against the oracle, to 1e-12: P equal to its transpose (each pair taken once) and not, at the
edges of the 4 rows and 256 columns of a workgroup and of the 32 x 32 tiles of the comparison with the transpose, in 1
to 4 dimensions, with the power and without, zeros in P, and points far apart."""
import numpy as np
import pytest

import fitsne_gpu as fg
import orc

pytestmark = pytest.mark.gpu


def kl(P, Y, df):
    c = fg.Context(no_dims=Y.shape[1], precision=fg.FP64_EXACT, df=df)
    c.set_P_dense(P)
    c.set_Y(Y)
    v = c.kl()
    c.close()
    return v


def dense_P(N, seed, symmetric):
    rng = np.random.default_rng(seed)
    P = rng.random((N, N)) ** 4
    P[rng.random((N, N)) < 0.3] = 0.0
    if symmetric:
        P = P + P.T
    np.fill_diagonal(P, 1e-9)
    return P / P.sum()


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("df", [1.0, 0.7])
@pytest.mark.parametrize("N,D", [(2, 2), (5, 1), (31, 2), (33, 3), (255, 2), (256, 4), (257, 2), (515, 1), (1030, 2)])
def test_kl(N, D, df, symmetric):
    print(f"[gpu] exact KL N={N} D={D} df={df} symmetric={symmetric}", flush=True)
    P = dense_P(N, N, symmetric)
    Y = np.random.default_rng(N + 7).normal(0, 5, size=(N, D))
    got, want = kl(P, Y, df), orc.exact_kl(P, Y, df=df)
    assert abs(got - want) <= 1e-12 * abs(want)


def test_one_asymmetric_entry():
    print("[gpu] exact KL, one entry differs", flush=True)
    P = dense_P(300, 1, True)
    P[299, 0] *= 1.5
    Y = np.random.default_rng(2).normal(0, 5, size=(300, 2))
    got, want = kl(P, Y, 1.0), orc.exact_kl(P, Y)
    assert abs(got - want) <= 1e-12 * abs(want)


@pytest.mark.parametrize("symmetric", [True, False])
def test_far_points(symmetric):
    print("[gpu] exact KL, far points", flush=True)
    P = dense_P(300, 3, symmetric)
    Y = np.random.default_rng(4).normal(0, 5, size=(300, 2))
    Y[7], Y[8] = 1e140, -1e90
    got, want = kl(P, Y, 1.0), orc.exact_kl(P, Y)
    assert abs(got - want) <= 1e-12 * abs(want)


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("df,N,D", [(1.0, 2047, 2), (1.0, 2048, 2), (0.7, 2049, 1), (1.0, 2079, 3), (0.7, 2081, 4)])
def test_kl_from_the_comparison_on(N, D, df, symmetric):
    """About 2,048 points: from there on P is compared with its transpose."""
    test_kl(N, D, df, symmetric)


@pytest.mark.parametrize("at", [(2099, 0), (2099, 2098), (31, 32), (0, 2099)])
def test_one_asymmetric_entry_of_many(at):
    print(f"[gpu] exact KL, entry {at} differs", flush=True)
    P = dense_P(2100, 1, True)
    P[at] = P[at] * 1.5 + 1e-4
    Y = np.random.default_rng(2).normal(0, 5, size=(2100, 2))
    got, want = kl(P, Y, 1.0), orc.exact_kl(P, Y)
    assert abs(got - want) <= 1e-12 * abs(want)


@pytest.mark.parametrize("symmetric", [True, False])
def test_far_points_over_the_triangle(symmetric):
    print("[gpu] exact KL, far points, triangle", flush=True)
    P = dense_P(2100, 3, symmetric)
    Y = np.random.default_rng(4).normal(0, 5, size=(2100, 2))
    Y[7], Y[8] = 1e140, -1e90
    got, want = kl(P, Y, 1.0), orc.exact_kl(P, Y)
    assert abs(got - want) <= 1e-12 * abs(want)
