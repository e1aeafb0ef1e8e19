"""Block steps of an ensemble against each cluster's own context, bit for bit
(precision "exact": the forces do not depend on the work plan): a few active
particles per block, and all of them (one lane per corrector); blocks of one
particle, cluster sizes around a block; a cluster that stops before the
others."""
import numpy as np
import pytest

from gravidy_amd import EnsembleHIP, Hermite4HIP, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu
SIZES = [1, 2, 255, 257, 1500, 512, 2049]


@pytest.mark.parametrize("dt_max", [0.125, 2.0 ** -14])
@pytest.mark.parametrize("t_end,steps", [(1.0, 1), (1.0, 7), (2.0 ** -12, 500)])
def test_ensemble_steps_are_the_clusters(dt_max, t_end, steps):
    systems = [ic.plummer(k, 11 + k) for k in SIZES]
    with EnsembleHIP(systems, E2, precision="exact", dt_max=dt_max) as e:
        e.set_small_path(0)
        e.init()
        info = e.run(t_end, t_end, steps)
        together = e.download()
    for (r, v), x, d in zip(systems, info, together):
        with Hermite4HIP(r, v, E2, precision="exact", dt_max=dt_max) as h:
            h.set_small_path(0)
            h.init_acc_jrk()
            atime = h.init_dt()
            one, _, _ = h.run(0.0, atime, t_end, t_end, steps)
            alone = h.download()
        assert (x["steps"], x["nsteps"], x["itime"]) == (one["steps"], one["nsteps"], one["itime"])
        for k in ("r", "v", "f", "t", "dt"):
            assert bits_equal(alone[k], d[k]), (r.shape[0], k)
