"""Copies between the caller's arrays and the device: sizes at the pieces and halves of the pinned buffer (256 KB, 1, 2
and 4 MB), with helper threads (8 MB and more) and odd remainders; the FP32 form's order and rounding; refused
values at either end, which leave the context as it was."""
import numpy as np
import pytest

import fitsne_gpu as fg

pytestmark = pytest.mark.gpu


def chain_P(N):
    row = np.arange(N + 1, dtype=np.uint32)
    col = ((np.arange(N) + 1) % N).astype(np.uint32)
    return row, col, np.full(N, 1.0 / N)


def fixed_order(Y):  # (2D: the min rule needs a coordinate below its predecessors)
    Y[0], Y[1] = 50.0, -50.0
    return Y


SIZES = [3, 1000, 16384, 16385, 65537, 131072, 131073, 262144 + 77, 700001, 1300003]


@pytest.mark.parametrize("D", [1, 2])
@pytest.mark.parametrize("N", SIZES)
def test_fp64_round_trip(N, D):
    print(f"[gpu] copies FP64 N={N} D={D}", flush=True)
    Y = fixed_order(np.random.default_rng(N).normal(size=(N, D)))
    c = fg.Context(no_dims=D, precision=fg.FP64_PLAIN)
    c.set_P(*chain_P(N))
    c.set_Y(Y)
    np.testing.assert_array_equal(c.get_Y().reshape(N, D), Y)
    for bad, at in ((np.nan, 0), (np.inf, N // 2), (-np.inf, N - 1)):
        Z = Y + 1.0
        Z[at, D - 1] = bad
        with pytest.raises(fg.FitsneError) as e:
            c.set_Y(Z)
        assert e.value.code == fg.E_ARG
    np.testing.assert_array_equal(c.get_Y().reshape(N, D), Y)
    c.close()


@pytest.mark.parametrize("D", [1, 2])
@pytest.mark.parametrize("N", SIZES)
def test_fp32_round_trip_and_gradient_order(N, D):
    print(f"[gpu] copies FP32 N={N} D={D}", flush=True)
    Y = fixed_order(np.random.default_rng(N + 1).normal(size=(N, D)))
    c = fg.Context(no_dims=D, precision=fg.FP32)
    c.set_P(*chain_P(N))
    c.set_Y(Y)
    np.testing.assert_array_equal(c.get_Y().reshape(N, D), Y.astype(np.float32).astype(np.float64))
    if N in (1000, 65537):  # the gradient in the caller's order: the FP64 form's, to the FP32 form's bound
        g = c.gradient()[0].reshape(N, D)
        r = fg.Context(no_dims=D, precision=fg.FP64_PLAIN)
        r.set_P(*chain_P(N))
        r.set_Y(Y.astype(np.float32).astype(np.float64))
        want = r.gradient()[0].reshape(N, D)
        r.close()
        assert np.linalg.norm(g - want) <= 1e-4 * np.linalg.norm(want)
    c.close()


@pytest.mark.parametrize("N,D,K", [(600, 30, 20), (3000, 60, 40), (40000, 60, 90)])
def test_knn_refuses_non_finite(N, D, K):
    print(f"[gpu] copies kNN N={N}", flush=True)
    X = np.random.default_rng(N).normal(size=(N, D))
    for at in (0, N * D - 1):
        Z = X.copy()
        Z.reshape(-1)[at] = np.inf
        with pytest.raises(fg.FitsneError) as e:
            fg.knn_exact(Z, K)
        assert e.value.code == fg.E_ARG
    idx, dist = fg.knn_exact(X, K)
    d = np.sqrt(((X[idx[-1]] - X[-1]) ** 2).sum(axis=1))
    np.testing.assert_allclose(dist[-1], d, rtol=1e-12)
    assert np.all(np.diff(dist[-1]) >= 0) and len(set(idx[-1])) == K


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nnz", [16383, 16385, 65535, 65537, 131071, 131073, 131137, 1 << 20, (1 << 20) + 1])
def test_small_P(nnz, prec):
    """P whose columns (4 bytes) and values (4 or 8) end about the first buffer's halves and end, and about the
    2^20 entries up to which the host converts them: the attractive term of every entry, by the gradient against the oracle."""
    print(f"[gpu] copies P nnz={nnz} {prec}", flush=True)
    import orc

    N = 2000
    rng = np.random.default_rng(nnz)
    row = np.r_[0, np.sort(rng.integers(0, nnz + 1, N - 1)), nnz].astype(np.uint32)
    col = rng.integers(0, N, nnz).astype(np.uint32)
    val = rng.random(nnz)
    val /= val.sum()
    Y = fixed_order(rng.normal(size=(N, 2)) * 12.0).astype(np.float32).astype(np.float64)
    c = fg.Context(no_dims=2, precision=fg.FP64_PLAIN if prec == "fp64" else fg.FP32)
    c.set_P(row, col, val)
    c.set_Y(Y)
    g, _ = c.gradient()
    c.close()
    want, _ = orc.gradient((row, col, val), Y)
    r = np.linalg.norm(g - want) / np.linalg.norm(want)
    assert r <= (1e-9 if prec == "fp64" else 1e-4), r


def test_contexts_copying_at_once():
    """Several threads, each with its own context and large copies, share the helper threads."""
    import threading

    N = 1300003
    print("[gpu] copies from four threads", flush=True)
    bad = []

    def work(k):
        try:
            Y = fixed_order(np.random.default_rng(k).normal(size=(N, 2)))
            c = fg.Context(no_dims=2, precision=fg.FP64_PLAIN)
            c.set_P(*chain_P(N))
            for r in range(3):
                c.set_Y(Y * (r + 1))
                if not np.array_equal(c.get_Y().reshape(N, 2), Y * (r + 1)):
                    bad.append((k, r))
            c.close()
        except Exception as e:  # (a thread's exception would not fail the test)
            bad.append((k, repr(e)))

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
