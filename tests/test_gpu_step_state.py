"""What follows h4h_step calls, whichever kernels made the steps: a loop that
goes on from the context's own block times (h4h_ensemble_run, h4h_tune_launch),
and the per-method calls, which find an empty active list."""
import numpy as np
import pytest

from gravidy_amd import EnsembleHIP, Hermite4HIP, _lib, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu


def _go_on(h, max_steps):
    info = _lib.H4HClusterInfo()
    _lib.check("h4h_ensemble_run", h.lib.h4h_ensemble_run(h._ctx, 1.0, 1.0, max_steps, info))
    return {k: getattr(info, k) for k, _ in info._fields_}


@pytest.mark.parametrize("precision", ["fp64", "mixed", "exact"])
@pytest.mark.parametrize("n", [300, 3000, 33000])
def test_loop_goes_on_from_single_steps(n, precision):
    """k steps one by one, then a loop of m: the loop of k + m."""
    k, m = 20, 3
    r, v = ic.plummer(n, 7 * n)
    with Hermite4HIP(r, v, E2, precision=precision) as h:
        h.init_acc_jrk()
        h.init_dt()
        whole = _go_on(h, k + m)
        want = h.download()
        h.upload(r, v)
        h.init_acc_jrk()
        a = h.init_dt()
        made = []
        for _ in range(k):
            c, a = h.step(a)
            made.append(c)
        first = _go_on(h, 1)
        assert first["steps"] == 1 and first["itime"] == a
        rest = _go_on(h, m - 1)
        assert rest["steps"] == m - 1
        assert sum(made) + first["nsteps"] + rest["nsteps"] == whole["nsteps"]
        assert (rest["itime"], rest["atime"]) == (whole["itime"], whole["atime"])
        got = h.download()
        for q in want:
            assert bits_equal(want[q], got[q]), q


@pytest.mark.parametrize("n", [300, 3000])
def test_one_cluster_ensemble_steps(n):
    """The same through an ensemble's handle of one cluster."""
    r, v = ic.plummer(n, n)
    with EnsembleHIP([(r, v)], E2) as e, Hermite4HIP(r, v, E2) as h:
        h.init_acc_jrk()
        a = h.init_dt()
        for _ in range(5):
            _, a = h.step(a)
        e.init()
        e.run(1.0, 1.0, 5)
        x, y = e.run(1.0, 1.0, 4)[0], _go_on(h, 4)
        assert x == y
        s, t = e.download()[0], h.download()
        for q in s:
            assert bits_equal(s[q], t[q]), q


@pytest.mark.parametrize("n", [300, 3000, 33000, 70000])
def test_active_list_is_empty_after_steps(n):
    r, v = ic.plummer(n, n + 1)
    with Hermite4HIP(r, v, E2) as h:
        h.init_acc_jrk()
        a = h.init_dt()
        for _ in range(40):
            assert h.find_particles_to_move(a) > 0
            for _ in range(2):
                last = a
                _, a = h.step(a)
            assert h.get_active().size == 0
            before = h.download()
            h.update_acc_jrk(0)
            h.correction_pos_vel(last, 0)
            after = h.download()
            for q in before:
                assert bits_equal(before[q], after[q]), q
