"""A team of workgroups that does not come together: the step is the launches',
and twice as many each time in a row up to 64, in loops, single steps and
across calls, with the same bits; then teams are tried again, and form."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP, _lib, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu


def _start(h, r, v):
    h.upload(r, v)
    h.init_acc_jrk()
    a = h.init_dt()
    h.team_steps(reset=True)
    return a


def _refuse(h):
    _lib.check("h4h_refuse_team", h.lib.h4h_refuse_team(h._ctx))


class Rule:
    """The steps a team makes, of active counts told one by one."""

    def __init__(self):
        self.rest = self.fails = self.made = 0

    def step(self, small, refused):
        """Whether a pending refusal is used up."""
        if self.rest:
            self.rest -= 1
        elif small and refused:
            self.rest = 2 ** min(self.fails, 6) - 1
            self.fails += 1
            return True
        elif small:
            self.made += 1
            self.fails = 0
        return False


def _settled(run):
    """run() until the counts it returns are as expected: a team may not form by
    itself after an idle time of the GPU (one in some hundred); it never makes
    more steps than expected."""
    for _ in range(6):
        got, want = run()
        assert got <= want
        if got == want:
            return
    assert got == want


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [1025, 3000, 32768, 40000])
def test_refused_teams(n, precision):
    limit = 128 if n > 32768 else 191 if precision == "mixed" else 256
    count = 150
    r, v = ic.plummer(n, n + 5)
    want = {}

    def same(h):
        s = h.download()
        for q in s:
            assert bits_equal(want.setdefault(q, s[q]), s[q]), q

    with Hermite4HIP(r, v, E2, precision=precision) as h:
        a = _start(h, r, v)
        sizes = h.run(0.0, a, 1.0, 1.0, count)[2]
        same(h)

        def loop():
            a = _start(h, r, v)
            _refuse(h)
            assert np.array_equal(h.run(0.0, a, 1.0, 1.0, count)[2], sizes)
            same(h)
            rule, refused = Rule(), True
            for k in sizes:
                refused &= not rule.step(k <= limit, refused)
            return h.team_steps(), rule.made

        def pieces(refusals):
            """Loops of one step: what is left alone is carried over."""
            a = _start(h, r, v)
            rule, refused, t = Rule(), False, 0.0
            for j, k in enumerate(sizes):
                if j < refusals:
                    _refuse(h)
                    refused = True
                info, _, n1 = h.run(t, a, 1.0, 1.0, 1)
                assert n1.tolist() == [k]
                t, a = info["itime"], info["atime"]
                refused &= not rule.step(k <= limit, refused)
            same(h)
            return h.team_steps(), rule.made

        def steps(refusals):
            a = _start(h, r, v)
            rule, refused = Rule(), False
            for j, k in enumerate(sizes):
                if j < refusals:
                    _refuse(h)
                    refused = True
                n1, a = h.step(a)
                assert n1 == k
                refused &= not rule.step(k <= 128, refused)
            same(h)
            return h.team_steps(), rule.made

        def both():
            """Single steps refused, then a loop, which leaves the rest alone."""
            a = _start(h, r, v)
            rule, refused, t = Rule(), False, 0.0
            for j, k in enumerate(sizes[:60]):
                _refuse(h)
                refused = True
                t, (_, a) = a, h.step(a)
                refused &= not rule.step(k <= 128, refused)
            h.run(t, a, 1.0, 1.0, count - 60)
            for k in sizes[60:]:
                refused &= not rule.step(k <= limit, refused)
            same(h)
            return h.team_steps(), rule.made

        _settled(loop)
        for refusals in (1, 8, 100):
            _settled(lambda: pieces(refusals))
            _settled(lambda: steps(refusals))
        _settled(both)
