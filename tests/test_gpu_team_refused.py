"""A team of workgroups that does not come together: the step and the 63 after
it are the launches', in loops, single steps and across calls, with the same
bits; then teams are tried again, and form."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP, _lib, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu
REST = 64


def _start(h, r, v):
    h.upload(r, v)
    h.init_acc_jrk()
    a = h.init_dt()
    h.team_steps(reset=True)
    return a


def _refuse(h):
    _lib.check("h4h_refuse_team", h.lib.h4h_refuse_team(h._ctx))


def _expected(k, limit):
    small = np.asarray(k) <= limit
    first = int(np.argmax(small))
    small[first:first + REST] = False
    return int(small.sum())


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [1025, 3000, 32768, 40000])
def test_refused_teams(n, precision):
    limit = 128 if n > 32768 else 191 if precision == "mixed" else 256
    r, v = ic.plummer(n, n + 5)
    with Hermite4HIP(r, v, E2, precision=precision) as h:
        a = _start(h, r, v)
        _, _, k = h.run(0.0, a, 1.0, 1.0, 150)
        assert h.team_steps() == (k <= limit).sum()
        want = h.download()
        # one loop
        a = _start(h, r, v)
        _refuse(h)
        _, _, k1 = h.run(0.0, a, 1.0, 1.0, 150)
        assert np.array_equal(k, k1) and h.team_steps() == _expected(k, limit)
        got = [h.download()]
        # loops of a few steps: the rest is carried over
        a = _start(h, r, v)
        _refuse(h)
        t, made = 0.0, 0
        while made < 150:
            info, _, _ = h.run(t, a, 1.0, 1.0, 10)
            t, a, made = info["itime"], info["atime"], made + info["steps"]
        assert h.team_steps() == _expected(k, limit)
        got.append(h.download())
        # single steps
        a = _start(h, r, v)
        _refuse(h)
        for x in k:
            y, a = h.step(a)
            assert x == y
        assert h.team_steps() == _expected(k, 128)
        got.append(h.download())
        # a single step refused, then loops
        a = _start(h, r, v)
        _refuse(h)
        t, made = 0.0, 0
        while not (k[made] <= 128):
            t, (_, a), made = a, h.step(a), made + 1
        t, (_, a), made = a, h.step(a), made + 1
        info, _, _ = h.run(t, a, 1.0, 1.0, REST - 1)
        assert info["steps"] == REST - 1 and h.team_steps() == 0
        info, _, _ = h.run(info["itime"], info["atime"], 1.0, 1.0, 150 - made - REST + 1)
        assert h.team_steps() == (k[made + REST - 1:] <= limit).sum()
        got.append(h.download())
        for s in got:
            for q in want:
                assert bits_equal(want[q], s[q]), q
