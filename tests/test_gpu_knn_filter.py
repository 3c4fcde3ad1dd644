"""The matrix-core filter behind fitsne_knn_mfma (N >= 1024) and fitsne_knn_exact (where it is faster), against
the oracle's VP-tree distances and against the FP64 kernel (reached with K = 257): the same neighbours and
distances, bit for bit.  Sizes at the edges of its tiles (32 points), workgroups (256 queries), chunks (16
coordinates, six of them the norms'), list lengths and thresholds; data far off centre, of extreme magnitude,
with repeated points and constant coordinates."""
import numpy as np
import pytest

import fitsne_gpu as fg
import orc

pytestmark = pytest.mark.gpu


def mixture(N, D, seed, k=12):
    rng = np.random.default_rng(seed)
    return rng.normal(0.0, 4.0, size=(k, D))[rng.integers(0, k, size=N)] + rng.normal(size=(N, D))


def check(X, K, got):
    idx, dist = got
    ridx, rdist = orc.knn_exact(X, K)
    assert np.array_equal(idx, ridx)
    assert np.array_equal(dist, rdist)


@pytest.mark.parametrize("N,D,K", [
    (1024, 10, 5), (1025, 11, 90), (1055, 26, 13), (1087, 42, 104), (1280, 58, 105), (1281, 74, 150), (1311, 90, 208),
    (1536, 106, 209), (1999, 122, 256), (2049, 128, 30), (3000, 1, 40), (3001, 2, 90)])
def test_filter_matches_the_oracle(N, D, K):
    X = mixture(N, D, N + D)
    print(f"[gpu] knn filter N={N} D={D} K={K}", flush=True)
    check(X, K, fg.knn_exact(X, K))
    check(X, K, fg.knn_mfma(X, K)[:2])


@pytest.mark.parametrize("N", [2, 33, 255, 256, 257, 511, 512, 513, 545, 1023])
def test_small_inputs_match_the_oracle(N):
    X = mixture(N, 7, N)
    K = min(N - 1, 200)
    print(f"[gpu] knn_mfma N={N} K={K}", flush=True)
    i, d, _ = fg.knn_mfma(X, K)
    check(X, K, (i, d))


@pytest.mark.parametrize("name", ["offset", "far", "tiny", "huge", "repeated", "constant", "one_axis", "all_equal"])
def test_filter_on_awkward_data(name):
    X = mixture(1500, 20, 3)
    if name == "offset":
        X = X + 1e6
    elif name == "far":  # centring leaves too few bits for the halves: the FP64 kernel takes it
        X = X + 1e12
    elif name == "tiny":
        X = X * 1e-170
    elif name == "huge":
        X = X * 1e150
    elif name == "repeated":
        X[700:1400] = X[:700]
    elif name == "constant":
        X[:, 5:] = 3.0
    elif name == "one_axis":
        X[:, 1:] *= 1e-7
    else:
        X[:] = X[0]
    print(f"[gpu] knn filter data={name}", flush=True)
    check(X, 45, fg.knn_mfma(X, 45)[:2])


@pytest.mark.parametrize("N,D,K", [(20011, 50, 90), (33000, 100, 150)])
def test_filter_matches_the_fp64_kernel(N, D, K):
    X = mixture(N, D, N, k=30)
    print(f"[gpu] knn filter N={N} D={D} K={K} against the FP64 kernel", flush=True)
    i_f, d_f, redo = fg.knn_mfma(X, K)
    i_e, d_e = fg.knn_exact(X, 257)
    assert np.array_equal(i_f, i_e[:, :K])
    assert np.array_equal(d_f, d_e[:, :K])
    assert redo <= N // 100


@pytest.mark.parametrize("name", ["cauchy", "half_equal", "most_equal", "ten_points", "one_far", "few_far", "lattice", "mass_and_rest", "thirty_places"])
@pytest.mark.parametrize("N", [1300, 4100])
def test_filter_where_queries_cannot_pass(name, N):
    """Thresholds within the error bound of zero distance, for all queries, for some of every workgroup, for whole
    workgroups: those go to the FP64 kernel, the others through the lists."""
    rng = np.random.default_rng(N)
    X = mixture(N, 12, N)
    if name == "cauchy":
        X = rng.standard_cauchy((N, 12))
    elif name == "half_equal":
        X[rng.random(N) < 0.5] = 1.0
    elif name == "most_equal":
        X[rng.random(N) < 0.97] = 1.0
    elif name == "ten_points":
        X = X[rng.integers(0, 10, N)]
    elif name == "one_far":
        X[5] *= 1e6
    elif name == "few_far":
        X[::100] *= 1e3
    elif name == "lattice":
        X = np.round(X[:, :3] / 3.0)
    elif name == "thirty_places":  # all at one distance from each other: every list overflows
        X = np.eye(30)[rng.integers(0, 30, N)]
    else:
        X[: N // 2] = X[0]  # whole workgroups of coinciding points, in front
    print(f"[gpu] knn filter {name} N={N}", flush=True)
    check(X, 40, fg.knn_mfma(X, 40)[:2])
    check(X, 40, fg.knn_exact(X, 40))


@pytest.mark.parametrize("N", [524288, 524289, 600001])
def test_queries_in_rounds(N):
    """As many queries as their lists are kept for at once (2^19), and more: the neighbours of some of every round,
    those at its ends among them, by distances added in coordinate order."""
    D, K = 3, 12
    X = mixture(N, D, N, k=40)
    print(f"[gpu] knn filter rounds N={N}", flush=True)
    idx, dist, redo = fg.knn_mfma(X, K)
    assert redo <= N // 100
    half = (N + 511) // 512 * 256
    for q in [0, 1, half - 1, half, half + 1, N - 257, N - 2, N - 1] + list(np.random.default_rng(1).integers(0, N, 40)):
        d2 = np.zeros(N)
        for d in range(D):
            d2 += (X[q, d] - X[:, d]) ** 2
        d2[q] = np.inf
        near = np.argpartition(d2, K + 8)[: K + 9]
        near = near[np.lexsort((near, d2[near]))][:K]
        assert np.array_equal(idx[q], near)
        assert np.array_equal(dist[q], np.sqrt(d2[near]))


@pytest.mark.parametrize("N,D,K", [
    (1024, 1, 33), (1024, 3, 64), (1100, 60, 65), (1400, 64, 65), (1407, 64, 65), (2999, 5, 70), (3000, 5, 70),
    (2188, 64, 21), (2187, 64, 21), (2000, 110, 20), (1999, 110, 20), (1500, 40, 32), (25000, 2, 8), (25000, 1, 8)])
def test_either_side_of_the_routes(N, D, K):
    """fitsne_knn_exact where it goes over from the FP64 kernel to the filter."""
    X = mixture(N, D, N + K)
    print(f"[gpu] knn_exact routes N={N} D={D} K={K}", flush=True)
    got = fg.knn_exact(X, K)
    if N <= 3000:
        check(X, K, got)
    i_e, d_e = fg.knn_exact(X, 257)
    assert np.array_equal(got[0], i_e[:, :K])
    assert np.array_equal(got[1], d_e[:, :K])
