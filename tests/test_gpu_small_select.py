"""Steps that the one-workgroup kernel leaves to the others, whose active
particles it selects itself, against the same steps selected by their own
launch: the states agree bit for bit and so does the step history.  Block
edges, blocks without active particles, all particles active."""
import numpy as np
import pytest

from gravidy_amd import EnsembleHIP, Hermite4HIP, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dt_max", [0.125, 2.0 ** -14])
@pytest.mark.parametrize("n", [2, 255, 256, 257, 700, 1024])
def test_steps_left_by_the_small_path(n, dt_max, precision):
    r, v = ic.plummer(n, n + 5)
    runs = []
    for act in (0, 1):
        with Hermite4HIP(r, v, E2, precision=precision, dt_max=dt_max) as h:
            h.set_small_path(act)
            h.init_acc_jrk()
            a = h.init_dt()
            info, t, k = h.run(0.0, a, 1.0, 1.0, 40)
            runs.append((info, t, k, h.download()))
    (i0, t0, k0, d0), (i1, t1, k1, d1) = runs
    # (steps of one particle are the one-workgroup kernel's own, with its own
    # order of the pair sums)
    if (k0 > 1).all():
        assert i0 == i1 and bits_equal(t0, t1) and (k0 == k1).all()
        for q in d0:
            assert bits_equal(d0[q], d1[q]), q
    else:
        j = int(np.argmin(k0 > 1))
        assert bits_equal(t0[: j + 1], t1[: j + 1]) and (k0[: j + 1] == k1[: j + 1]).all()


@pytest.mark.parametrize("steps", [1, 9])
def test_clusters_left_by_the_small_path(steps):
    systems = [ic.plummer(k, k) for k in (2, 1024, 256, 255, 513)]
    runs = []
    for act in (0, 1):
        with EnsembleHIP(systems, E2, dt_max=2.0 ** -14) as e:
            e.set_small_path(act)
            e.init()
            runs.append((e.run(1.0, 1.0, steps), e.download()))
    assert runs[0][0] == runs[1][0]
    for a, b in zip(runs[0][1], runs[1][1]):
        for q in a:
            assert bits_equal(a[q], b[q]), q
