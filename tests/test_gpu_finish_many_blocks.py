"""Block steps of ensembles around the number of blocks from which the finish is
two passes, against the clusters alone: bit for bit in exact precision (the
forces do not depend on the work plan), the schedule and the state to rounding
in the others."""
import numpy as np
import pytest

from gravidy_amd import EnsembleHIP, Hermite4HIP, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu
SOME = [1, 2, 255, 257, 1500, 512, 2049]  # 22 blocks


def _alone(r, v, precision, dt_max, t_end, steps):
    with Hermite4HIP(r, v, E2, precision=precision, dt_max=dt_max) as h:
        h.set_small_path(0)
        h.init_acc_jrk()
        atime = h.init_dt()
        info, _, _ = h.run(0.0, atime, t_end, t_end, steps)
        return info, h.download()


@pytest.mark.parametrize("precision,dt_max,steps", [("exact", 2.0 ** -14, 7), ("exact", 0.125, 40),
                                                    ("fp64", 2.0 ** -14, 7), ("fp64", 0.125, 40),
                                                    ("mixed", 2.0 ** -14, 7)])
@pytest.mark.parametrize("pairs", [1013, 1014, 1500])  # 2048, 2050 and 3022 blocks
def test_steps_are_the_clusters(precision, dt_max, steps, pairs):
    small = [ic.plummer(300, k) for k in range(4)]  # 2 blocks each
    systems = [ic.plummer(k, 11 + k) for k in SOME] + [small[k % 4] for k in range(pairs)]
    t_end = 2.0 ** -12 if steps > 7 else 1.0
    with EnsembleHIP(systems, E2, precision=precision, dt_max=dt_max) as e:
        e.init()
        info = e.run(t_end, t_end, steps)
        together = e.download()
    for c in list(range(len(SOME))) + [len(SOME), len(systems) - 1]:
        r, v = systems[c]
        one, alone = _alone(r, v, precision, dt_max, t_end, steps)
        assert (info[c]["steps"], info[c]["nsteps"], info[c]["itime"], info[c]["atime"]) == (
            one["steps"], one["nsteps"], one["itime"], one["atime"])
        for k in ("r", "v", "f", "t", "dt"):
            x, y = together[c][k], alone[k]
            if precision == "exact" or k in ("t", "dt"):
                assert bits_equal(x, y), (c, k)
            elif precision == "fp64" or k != "f":
                # sums in another order: 2^-53 sqrt(n) or so of the largest term
                # a step, 2^-24 of it in the FP32 runs
                tol = 1e-10 if precision == "fp64" else 1e-6
                assert np.abs(x - y).max() <= tol * max(1.0, np.abs(y).max()), (c, k)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_small_clusters_are_the_same_in_more_company(precision):
    """Clusters with a workgroup of their own, 2000 blocks and 2200: the plan of
    a cluster of two tiles does not depend on the others, so the bits agree."""
    small = [ic.plummer(300, k) for k in range(5)]
    out = []
    for count in (1000, 1100):
        with EnsembleHIP([small[k % 5] for k in range(count)], E2, precision=precision) as e:
            e.init()
            info = e.run(2.0 ** -7, 2.0 ** -7)
            assert e.stats()["small_steps"] > 0
            out.append((info, e.download()))
    (a, s), (b, t) = out
    assert sum(x["steps"] for x in a) > 0
    for c in (0, 1, 2, 3, 4, 999):
        assert a[c] == b[c] == b[1000 + c % 5]
        for k in s[c]:
            assert bits_equal(s[c][k], t[c][k]), (c, k)
            assert bits_equal(s[c][k], t[1000 + c % 5][k]), (c, k)
