"""The ordered Z sum of the Barnes-Hut path (fitsne_seqsum.hpp), run by a CPU emulation of its workgroup,
against a loop that adds in index order: equal bit for bit, and it ends, also where the running sum is zero, tiny,
huge or not finite, in front, in between and over several wavefronts and chunks (16 values a thread, 1024 a
wavefront, 16,384 a chunk)."""
import os
import struct
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("seqsum") / "seqsum_host")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas", "-o", exe,
                    os.path.join(HERE, "seqsum_host.cpp")], check=True)
    return exe


def values(name):
    rng = np.random.default_rng(5)
    q = rng.random(3000) * 40.0
    if name == "one":
        return np.array([3.5])
    if name == "usual":
        return rng.random(40001) * 40.0
    if name == "ties":  # halves of an ulp once the sum is large
        return np.r_[2.0 ** 52, np.full(2000, 0.5), np.full(2000, 1.5)]
    if name == "zeros":
        return np.zeros(100)
    if name == "zeros_many":
        return np.zeros(20000)
    if name == "zeros_first":
        return np.r_[np.zeros(1100), q]
    if name == "tiny":
        return np.full(40, 1e-260)
    if name == "tiny_to_range":  # from below the range into it
        return np.full(2000, 1e-252)
    if name == "subnormal":
        return np.full(1500, 5e-324)
    if name == "tiny_then_usual":
        return np.r_[np.full(1030, 1e-300), q]
    if name == "huge":
        return np.full(300, 1e260)
    if name == "overflow":
        return np.r_[q, np.full(300, 1e308)]
    if name == "inf":
        return np.r_[q, np.inf, q]
    if name == "nan_first":
        return np.r_[np.nan, q]
    if name == "nan_behind":
        return np.r_[q, np.nan, q]
    assert name == "negative"
    return np.r_[q, -q[:40], q]


@pytest.mark.parametrize("name", ["one", "usual", "ties", "zeros", "zeros_many", "zeros_first", "tiny", "tiny_to_range",
                                  "subnormal", "tiny_then_usual", "huge", "overflow", "inf", "nan_first", "nan_behind",
                                  "negative"])
def test_ordered_sum(harness, name):
    v = values(name)
    with np.errstate(all="ignore"):
        want = np.cumsum(v)[-1]  # in order, one rounding an addition
        inv = np.float64(1.0) / want
    r = subprocess.run([harness], input=struct.pack("<q", len(v)) + v.tobytes(), capture_output=True, timeout=100)
    assert r.returncode == 0, r.stdout.decode()
    got = [struct.unpack("<d", struct.pack("<Q", int(x, 16)))[0] for x in r.stdout.split()]
    for g, w in zip(got, (want, inv)):
        assert g == w or (np.isnan(g) and np.isnan(w))
