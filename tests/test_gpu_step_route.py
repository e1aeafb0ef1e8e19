"""Consecutive h4h_step calls, which skip the kernels for small steps when the
step before has counted a larger one, against the device loop (the same bits),
also when the state changes between two steps."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu


def steps(h, atime, count):
    times, counts = [], []
    for _ in range(count):
        times.append(atime)
        k, atime = h.step(atime)
        counts.append(k)
    return np.array(times), np.array(counts), atime


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [300, 1024, 1025, 6000, 33000])
def test_steps_are_the_device_loops(n, precision):
    r, v = ic.plummer(n, 3 * n)
    with Hermite4HIP(r, v, E2, precision=precision) as h:
        h.init_acc_jrk()
        a = h.init_dt()
        info, t, k = h.run(0.0, a, 1.0, 1.0, 150)
        run = h.download()
        h.upload(r, v)
        h.init_acc_jrk()
        assert h.init_dt() == a
        t1, k1, a1 = steps(h, a, 150)
        one = h.download()
        assert bits_equal(t, t1) and (k == k1).all() and a1 == info["atime"]
        for q in run:
            assert bits_equal(run[q], one[q]), q
        # another state at the time of the step that the last one counted
        assert (k1 > 128).any()
        f, tt = one["f"].copy(), one["t"].copy()
        dt = np.full(n, 2.0 ** -3)
        dt[5] = 2.0 ** -6
        h.upload(r, v, f, np.full(n, a1 - 2.0 ** -6), dt)
        assert h.step(a1)[0] == 1
        after = h.download()
        h.upload(r, v, f, np.full(n, a1 - 2.0 ** -6), dt)
        h.run(-1.0, a1, 10.0, -1.0, 1)
        again = h.download()
        for q in after:
            assert bits_equal(after[q], again[q]), q
