"""Active sets around the most that one workgroup per tile takes (256 with one
tile each, 128 with two and in a single h4h_step), all in one tile or spread
over all of them, against the same step on the selection, update and finish
launches: the same bits, in the device loop and by h4h_step."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP

from test_gpu_parity import E2, bits_equal, block_state

pytestmark = pytest.mark.gpu
T1 = 1.0 + 2.0 ** -12


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n,nact,spread", [
    (1025, 129, 1), (1025, 256, 1), (1025, 256, 4), (1025, 257, 4), (3000, 144, 11),
    (3000, 145, 2), (9000, 191, 35), (9000, 192, 1), (32768, 255, 127), (32768, 256, 128),
    (32768, 257, 128), (40000, 128, 156), (40000, 129, 1)])
def test_team_sets_up_to_the_largest(n, nact, spread, prec):
    r, v, f, t, dt = block_state(n, n + nact, T1)
    rng = np.random.default_rng(n + nact)
    dt[:] = 2.0 ** -rng.integers(3, 10, size=n).astype(float)
    t[:] = 1.0
    tiles = rng.choice(n // 256, size=spread, replace=False)
    pool = np.concatenate([256 * b + np.arange(256) for b in tiles])
    dt[rng.choice(pool, size=nact, replace=False)] = 2.0 ** -12
    out = []
    for how in ("others", "loop", "step"):
        with Hermite4HIP(r, v, E2, precision=prec) as h:
            if how == "others":
                h.set_tuning({})
            h.upload(r, v, f, t, dt)
            if how == "step":
                k1, a = h.step(T1)
                k2, a = h.step(a)
                sn = [k1, k2]
            else:
                info, _, sn = h.run(1.0, T1, 2.0, 2.0, 2)
                a = info["atime"]
            out.append((list(sn), a, h.download()))
    assert out[0][0][0] == nact
    for k, a, s in out[1:]:
        assert k == out[0][0] and a == out[0][1]
        for q in s:
            assert bits_equal(s[q], out[0][2][q]), q
