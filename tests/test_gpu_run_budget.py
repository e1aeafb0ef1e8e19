"""Device loops that end with their step budget (the last steps enqueued with
their own loop tail) against one `h4h_step` per step: the same bits, history
and counters for budgets around a captured chunk of 32 steps, and when the
loop stops before the budget is spent."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu


def start(h, r, v):
    h.upload(r, v)
    h.init_acc_jrk()
    return h.init_dt()


@pytest.mark.parametrize("n,precision", [(300, "exact"), (66000, "fp64")])
@pytest.mark.parametrize("budget", [1, 31, 32, 33, 64, 65])
@pytest.mark.parametrize("graphs", [True, False])
def test_budget_around_a_chunk(n, precision, budget, graphs):
    r, v = ic.plummer(n, n)
    with Hermite4HIP(r, v, E2, precision=precision) as h:
        h.set_graphs(graphs)
        a = start(h, r, v)
        info, t, k = h.run(0.0, a, 1.0, 1.0, budget)
        run = h.download()
        # the loop goes on from there as one step after the other
        info2, t2, k2 = h.run(info["itime"], info["atime"], 1.0, 1.0, 3)
        a1 = start(h, r, v)
        t1, k1 = [], []
        for _ in range(budget):
            t1.append(a1)
            m, a1 = h.step(a1)
            k1.append(m)
        one = h.download()
    assert info["steps"] == budget and info["atime"] == a1 and info["last_nact"] == k1[-1]
    assert info["nsteps"] == sum(k1) and info["interactions"] == n * sum(k1)
    assert bits_equal(t, np.array(t1)) and list(k) == k1
    assert info2["steps"] == 3 and t2[0] == a1
    for q in run:
        assert bits_equal(run[q], one[q]), q


@pytest.mark.parametrize("graphs", [True, False])
def test_stop_before_the_budget(graphs):
    r, v = ic.plummer(300, 300)
    with Hermite4HIP(r, v, E2, precision="exact") as h:
        h.set_graphs(graphs)
        a = start(h, r, v)
        _, t, k = h.run(0.0, a, 1.0, 1.0, 12)
        a = start(h, r, v)
        info, ts, ks = h.run(0.0, a, 1.0, t[4], 20)
    assert info["steps"] == 5 and bits_equal(ts, t[:5]) and (ks == k[:5]).all()
    assert info["itime"] == t[4] and info["atime"] == t[5]
