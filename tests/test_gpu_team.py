"""Block steps made by one workgroup per j tile (systems of 5 to 256 tiles)
against the same steps on the selection, update and finish launches: the
same bits, whichever makes a step.  An empty tuning table keeps the default
plans but turns the former off."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP, ic

from test_gpu_parity import E2, bits_equal, block_state

pytestmark = pytest.mark.gpu


def _run(r, v, prec, steps, team, mode="run", graphs=True):
    with Hermite4HIP(r, v, E2, precision=prec) as h:
        if not team:
            h.set_tuning({})
        h.set_graphs(graphs)
        res = h.integration(1.0, interval=1.0, max_steps=steps, mode=mode)
        p, _ = h.download_predictor()
        return res, h.download(), p


def _same(a, b):
    (ra, sa, pa), (rb, sb, pb) = a, b
    assert np.array_equal(ra["step_time"], rb["step_time"])
    assert np.array_equal(ra["step_nact"], rb["step_nact"])
    for k in ("r", "v", "f", "t", "dt", "old", "a2", "a3"):
        assert bits_equal(sa[k], sb[k]), k
    assert bits_equal(pa, pb)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n,steps", [(1025, 300), (1280, 64), (2048, 200), (2049, 100), (5000, 200),
                                     (8192, 100), (8193, 100), (16384, 60), (16385, 60),
                                     (32768, 40), (32769, 40), (65536, 40)])
def test_team_steps_are_the_other_steps_bits(prec, n, steps):
    r, v = ic.plummer(n, 60 + n)
    _same(_run(r, v, prec, steps, True), _run(r, v, prec, steps, False))


@pytest.mark.parametrize("n", [1500, 10007])
def test_team_loop_modes_agree(n):
    r, v = ic.plummer(n, 3)
    one = _run(r, v, "fp64", 120, True)
    _same(one, _run(r, v, "fp64", 120, True, graphs=False))
    _same(one, _run(r, v, "fp64", 120, True, mode="step"))


T1 = 1.0 + 2.0 ** -12


@pytest.mark.parametrize("n,nact,spread", [(3000, 1, 1), (3000, 4, 1), (3000, 13, 2), (3000, 47, 1),
                                           (3000, 48, 11), (3000, 64, 3), (3000, 65, 11),
                                           (9000, 96, 1), (9000, 127, 30), (9000, 128, 1),
                                           (9000, 128, 35), (9000, 129, 2), (20000, 128, 78),
                                           (20000, 100, 2)])
def test_team_step_active_set_edges(n, nact, spread):
    """nact active particles in `spread` tiles, 128 the most a team takes;
    two steps, the second of whatever comes next."""
    r, v, f, t, dt = block_state(n, n + nact, T1)
    rng = np.random.default_rng(n + nact)
    dt[:] = 2.0 ** -rng.integers(3, 10, size=n).astype(float)
    t[:] = 1.0
    tiles = rng.choice((n + 255) // 256 - 1, size=spread, replace=False)
    pool = np.concatenate([256 * b + np.arange(256) for b in tiles])
    dt[rng.choice(pool, size=nact, replace=False)] = 2.0 ** -12
    out = []
    for team in (True, False):
        with Hermite4HIP(r, v, E2, precision="fp64") as h:
            if not team:
                h.set_tuning({})
            h.upload(r, v, f, t, dt)
            info, st, sn = h.run(1.0, T1, 2.0, 2.0, 2)
            assert sn[0] == nact
            out.append(({"step_time": st, "step_nact": sn}, h.download(), h.download_predictor()[0]))
    _same(*out)


def test_team_leaves_times_within_the_tolerance_to_the_others():
    n = 4000
    r, v, f, t, dt = block_state(n, 9, T1)
    dt[:] = 2.0 ** -5
    t[:] = 1.0
    dt[[5, 700]] = 2.0 ** -12
    t2 = T1 + 2.0 ** -13
    a, b = [300, 301, 900], [302, 1000, 3999]
    t[a + b] = 0.0
    dt[a] = t2
    dt[b] = np.nextafter(t2, 2.0)
    out = []
    for team in (True, False):
        with Hermite4HIP(r, v, E2, precision="fp64", dt_min=2.0 ** -12) as h:
            if not team:
                h.set_tuning({})
            h.upload(r, v, f, t, dt)
            info, st, sn = h.run(1.0, T1, 2.0, 2.0, 2)
            assert sn.tolist() == [2, 6]
            out.append(({"step_time": st, "step_nact": sn}, h.download(), h.download_predictor()[0]))
    _same(*out)


def test_two_systems_at_once_on_two_threads():
    """Two threads drive a system each on the same GPU: their teams form or
    do not, with the same bits as alone."""
    import threading
    cases = [(10007, "fp64", 150), (33000, "fp64", 80), (5000, "mixed", 200)]
    sys_ = [ic.plummer(n, n) for n, _, _ in cases]
    alone = [_run(r, v, p, k, True) for (r, v), (_, p, k) in zip(sys_, cases)]
    got = [None] * len(cases)

    def work(j):
        (r, v), (_, p, k) = sys_[j], cases[j]
        got[j] = _run(r, v, p, k, True)

    threads = [threading.Thread(target=work, args=(j,)) for j in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, got):
        _same(a, b)
