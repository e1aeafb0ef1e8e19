"""Which block steps one workgroup per j tile or two makes (h4h_team_steps): all
with up to the documented number of active particles, and no others, so that
tests that compare them with the launches' do compare two things."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP, ic

from test_gpu_parity import E2, block_state

pytestmark = pytest.mark.gpu
T1 = 1.0 + 2.0 ** -12


def _largest(n, precision, one):
    if one or n > 32768:
        return 128
    return 191 if precision == "mixed" else 256


def _settled(run):
    """run() until the counts it returns are as expected: a team may not form
    after an idle time of the GPU (one in some hundred), and its step is then the
    launches'; it never makes more steps than expected."""
    for _ in range(6):
        got, want = run()
        assert got <= want
        if got == want:
            return
    assert got == want


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,steps", [(1025, 200), (2048, 200), (5000, 200), (10007, 200),
                                     (32768, 100), (32769, 100), (50000, 100)])
def test_the_small_steps_are_its(n, steps, precision):
    r, v = ic.plummer(n, 60 + n)
    with Hermite4HIP(r, v, E2, precision=precision) as h:

        def run(mode):
            h.upload(r, v)
            h.team_steps(reset=True)
            k = h.integration(1.0, interval=1.0, max_steps=steps, mode=mode)["step_nact"]
            want = (k <= _largest(n, precision, mode == "step")).sum()
            assert want > 0 and (k > 256).any()
            return h.team_steps(), want

        for mode in ("run", "step"):
            _settled(lambda: run(mode))
        for off in (lambda: h.set_tuning({}), lambda: (h.set_tuning(None), h.set_precision("exact"))):
            off()
            for mode in ("run", "step"):
                assert run(mode)[0] == 0


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [1025, 9000, 32768, 40000])
def test_set_sizes(n, precision):
    for nact in (1, 64, 127, 128, 129, 191, 192, 255, 256, 257):
        r, v, f, t, dt = block_state(n, n + nact, T1)
        rng = np.random.default_rng(n + nact)
        dt[:] = 2.0 ** -5
        t[:] = 1.0
        dt[rng.choice(n, size=nact, replace=False)] = 2.0 ** -12
        with Hermite4HIP(r, v, E2, precision=precision) as h:

            def run(one):
                h.upload(r, v, f, t, dt)
                h.team_steps(reset=True)
                if one:
                    assert h.step(T1)[0] == nact
                else:
                    assert h.run(1.0, T1, 2.0, 2.0, 1)[2].tolist() == [nact]
                return h.team_steps(), int(nact <= _largest(n, precision, one))

            for one in (False, True):
                _settled(lambda: run(one))
