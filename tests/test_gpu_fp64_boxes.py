"""The FP64 path's stages in box order (counting sort, spread per box and wavefront, interpolation) against the
oracle, to the FP64 path's bound of 1e-9: the edges of the 64-point wavefronts and 256-point workgroups, one point to
a box, all but the corners in one box, 2 to 5 nodes per box, more boxes than one tile of the offsets' scan (16384)."""
import numpy as np
import pytest

import fitsne_gpu as fg
import orc
from datagen import blobs, random_csr

pytestmark = pytest.mark.gpu
TOL = 1e-9


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


def compare(Y, df, p=3, mni=50):
    N, D = Y.shape
    P = random_csr(N, min(6, N - 1), seed=N + D)
    c = fg.Context(no_dims=D, precision=fg.FP64_PLAIN, df=df, n_interpolation_points=p, min_num_intervals=mni)
    try:
        c.set_P(*P)
        c.set_Y(Y)
        got, z = c.gradient()
        again, z2 = c.gradient()  # the counters are clear again
    finally:
        c.close()
    want, zw = orc.gradient(P, Y, p=p, min_num_intervals=mni, df=df)
    print(f"    rel={rel(got, want):.2e} Zrel={abs(z - zw) / abs(zw):.2e}", flush=True)
    assert rel(got, want) <= TOL and rel(again, want) <= TOL
    assert abs(z - zw) <= TOL * abs(zw) and abs(z2 - zw) <= TOL * abs(zw)


@pytest.mark.parametrize("df", [1.0, 0.6])
@pytest.mark.parametrize("D", [1, 2])
@pytest.mark.parametrize("N", [5, 63, 64, 65, 127, 255, 256, 257, 4099])
def test_edges(N, D, df):
    print(f"[gpu] fp64 boxes N={N} D={D} df={df}", flush=True)
    compare(blobs(N, D, 4, seed=N, span=30.0, sd=2.0), df)


@pytest.mark.parametrize("df", [1.0, 0.6])
@pytest.mark.parametrize("D", [1, 2])
@pytest.mark.parametrize("p", [2, 3, 4, 5])
def test_nodes_per_box(p, D, df):
    print(f"[gpu] fp64 boxes p={p} D={D} df={df}", flush=True)
    compare(blobs(1500, D, 5, seed=p, span=30.0, sd=2.0), df, p=p)


@pytest.mark.parametrize("name", ["one_per_box", "one_box", "many_boxes"])
@pytest.mark.parametrize("D", [1, 2])
def test_boxes(name, D):
    print(f"[gpu] fp64 boxes {name} D={D}", flush=True)
    rng = np.random.default_rng(D)
    mni = 50
    if name == "one_per_box":
        t = (np.arange(50) + 0.5) / 50 * 40 - 20
        Y = t[:, None] if D == 1 else np.stack(np.meshgrid(t, t), -1).reshape(-1, 2)
        Y = Y[rng.permutation(len(Y))]
    elif name == "one_box":
        Y = rng.uniform(10.05, 10.35, size=(1000, D))
        Y = Y[np.argsort(-Y[:, 0])]  # (2D: the min rule needs a decreasing coordinate)
        Y[0], Y[1] = 25.0, -25.0
    else:
        mni = 131 if D == 2 else 600  # (1D: an FFT of at most 4096)
        Y = rng.normal(0, 8, size=(3000, D))
    compare(Y, 1.0, mni=mni)


@pytest.mark.parametrize("per", [61, 6])
@pytest.mark.parametrize("D", [1, 2])
def test_streams(D, per):
    """Both sides of the six million entries from which the step runs on three streams: the gradient against the
    oracle, and three steps with overlap on against those with it off (atomics add in any order)."""
    N = 100_001
    print(f"[gpu] fp64 streams D={D} per={per}", flush=True)
    P = random_csr(N, per, seed=per, symmetric=False)
    Y = blobs(N, D, 8, seed=D, span=30.0, sd=2.0)
    out = []
    for overlap in (True, False):
        c = fg.Context(no_dims=D, precision=fg.FP64_PLAIN)
        c.set_overlap(overlap)
        c.set_P(*P)
        c.set_Y(Y)
        g, z = c.gradient()
        for _ in range(3):
            c.step(0.5, 200.0, 5.0)
        out.append((g, z, c.get_Y()))
        c.close()
    want, zw = orc.gradient(P, Y)
    for g, z, y in out:
        assert rel(g, want) <= TOL and abs(z - zw) <= TOL * abs(zw)
        assert rel(y, out[0][2]) <= TOL
