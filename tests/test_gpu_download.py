"""h4h_download (written by the device into pinned slots and copied on by one
or more threads) against the arrays downloaded one at a time and against what
was uploaded, bit for bit: one double below and above the 4 MB of larger slots
and more threads, pieces that end inside an array, a ragged last piece,
clusters back to back."""
import ctypes

import numpy as np
import pytest

from gravidy_amd import EnsembleHIP, Hermite4HIP, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu
ROWS = {"r": 4, "v": 4, "f": 6, "t": 1, "dt": 1, "old": 6, "a2": 3, "a3": 3}


def download(h, n, names):
    out = {k: np.full((n, ROWS[k]), 7.25) for k in names}
    ptr = lambda k: out[k].ctypes.data_as(ctypes.POINTER(ctypes.c_double)) if k in out else None
    assert h.lib.h4h_download(h._ctx, *(ptr(k) for k in ROWS)) == 0
    return out


def check(h, n, given):
    every = download(h, n, ROWS)
    for k in ROWS:
        assert bits_equal(every[k], download(h, n, [k])[k]), k
    for k, a in given.items():
        assert bits_equal(every[k].reshape(a.shape), a), k
    # a subset: other places of the same arrays in the pieces
    some = download(h, n, ["v", "old", "a3", "dt"])
    for k in some:
        assert bits_equal(every[k], some[k]), k


# 28 doubles per particle: 524288 doubles are 4 MB
@pytest.mark.parametrize("n", [18724, 18725, 32768, 100003, 150000])
def test_large_download(n):
    rng = np.random.default_rng(n)
    r, v = ic.plummer(n, n)
    f = rng.normal(size=(n, 6))
    t = np.zeros(n)
    dt = 2.0 ** -rng.integers(3, 8, size=n).astype(float)
    with Hermite4HIP(r, v, E2) as h:
        h.upload(r, v, f, t, dt)
        v4 = v.copy()
        v4[:, 3] = 0.0
        check(h, n, {"r": r, "v": v4, "f": f, "t": t, "dt": dt})
        h.step(2.0 ** -7)  # old, a2, a3 of the active particles
        check(h, n, {})


# one piece, a piece more than one and two (32768 doubles), the second thread's
@pytest.mark.parametrize("n", [1, 2, 300, 1170, 1171, 2340, 2341, 9000])
def test_small_download(n):
    r, v = ic.plummer(n, n)
    f = np.random.default_rng(n).normal(size=(n, 6))
    t = np.zeros(n)
    dt = np.full(n, 2.0 ** -5)
    with Hermite4HIP(r, v, E2) as h:
        h.upload(r, v, f, t, dt)
        check(h, n, {"r": r, "f": f, "t": t, "dt": dt})
        h.step(2.0 ** -5)
        check(h, n, {})


def test_large_download_of_clusters():
    sizes = [1, 255, 256, 9000, 257, 20001]
    systems = [ic.plummer(k, 3 + k) for k in sizes]
    with EnsembleHIP(systems, E2) as e:
        r = np.concatenate([s[0] for s in systems])
        check(e, sum(sizes), {"r": r})
