"""One-workgroup block steps at the edges of their lane layout (8 corrector
lanes per active slot, slots rounded up to a power of two, 64 and more slots
on whole waves, two particles per thread), and next block times within
find_particles_to_move's tolerance of each other."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP

from test_gpu_parity import E2, bits_equal, block_state

pytestmark = pytest.mark.gpu

T1 = 1.0 + 2.0 ** -12


def _state(n, nact, seed):
    """A state with exactly nact particles active at T1."""
    rng = np.random.default_rng(seed)
    r, v, f, t, dt = block_state(n, seed, T1) if n > 1 else (
        np.array([[0.1, 0.2, 0.3, 1.0]]), np.array([[0.3, 0.2, 0.1, 0.0]]),
        rng.normal(size=(1, 6)), np.zeros(1), np.zeros(1))
    pick = rng.choice(n, size=nact, replace=False)
    dt[:] = 2.0 ** -rng.integers(3, 10, size=n).astype(float)
    t[:] = 1.0
    dt[pick] = 2.0 ** -12
    return r, v, f, t, dt, np.sort(pick).astype(np.uint32)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [300, 512, 513, 1024])
@pytest.mark.parametrize("nact", [1, 2, 7, 8, 9, 16, 31, 32, 33, 63, 64, 65, 127, 128, 129, 200,
                                  255, 256])
def test_small_step_slot_edges(oracle, prec, n, nact):
    r, v, f, t, dt, mo = _state(n, nact, 7 * n + nact)
    with Hermite4HIP(r, v, E2, precision=prec) as h:
        h.set_small_path(256)
        h.upload(r, v, f, t, dt)
        h.stats(reset=True)
        k, atime = h.step(T1)
        assert h.stats()["small_steps"] == 1
        s = h.download()
    with Hermite4HIP(r, v, E2, precision=prec) as h:
        h.set_small_path(0)
        h.upload(r, v, f, t, dt)
        k2, atime2 = h.step(T1)
        m = h.download()
    assert k == k2 == nact and atime == atime2
    assert bits_equal(s["old"][mo], f[mo])
    # the multi-workgroup step sums the same pairs in another order
    scale = np.abs(m["f"]).max()
    assert np.abs(s["f"] - m["f"]).max() <= (1e-12 if prec == "fp64" else 2e-6) * scale
    # the corrector is the oracle's, bit for bit, on the forces the step made
    po, _ = oracle.predicted_pos_vel(T1, t, r, v, f)
    z3 = np.zeros((n, 3))
    a2, a3, rc, vc, tc, dtc = oracle.correction_pos_vel(T1, mo, po, s["f"], f, z3, z3, r, v, t, dt)
    assert bits_equal(s["r"][:, :3], rc[:, :3]) and bits_equal(s["v"][:, :3], vc[:, :3])
    assert bits_equal(s["a2"][mo], a2[mo]) and bits_equal(s["a3"][mo], a3[mo])
    assert bits_equal(s["t"], tc) and bits_equal(s["dt"], dtc)


@pytest.mark.parametrize("n,nact", [(600, 1), (600, 40), (1024, 90)])
def test_small_loop_joins_times_within_the_tolerance(n, nact):
    """Times one rounding apart (closer than the selection's tolerance of
    2 DBL_EPSILON) are one block: the next step after T1 moves both groups."""
    r, v, f, t, dt, mo = _state(n, nact, n)
    t2 = T1 + 2.0 ** -13
    rest = np.setdiff1d(np.arange(n), mo)
    a, b = rest[:3], rest[3:8]
    t[a] = t[b] = 0.0
    dt[a] = t2
    dt[b] = np.nextafter(t2, 2.0)
    assert 0 < dt[b[0]] - t2 < 2 * np.finfo(float).eps
    out = []
    for limit in (256, 0):
        # (dt_min 2^-12: the particles moved at T1 come after t2)
        with Hermite4HIP(r, v, E2, precision="fp64", dt_min=2.0 ** -12) as h:
            h.set_small_path(limit)
            h.upload(r, v, f, t, dt)
            h.stats(reset=True)
            info, st, sn = h.run(1.0, T1, 2.0, 2.0, 2)
            out.append((st.tolist(), sn.tolist(), info["atime"], h.stats()["small_steps"]))
    assert out[0][:3] == out[1][:3]
    assert out[0][3] == 2 and out[1][3] == 0
    assert out[0][1] == [nact, 8]
