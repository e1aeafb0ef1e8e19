"""Exact forces of ensembles, a lane per particle or a few per workgroup: the
bits of each cluster alone."""
import pytest

from gravidy_amd import EnsembleHIP, Hermite4HIP, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[64] * 900, [700] * 70, [1025, 1024, 1, 257] * 40,
                                   [300] * 8, [9000, 20000, 3], [2, 500, 257, 1025, 4000]])
def test_forces_and_steps_are_each_clusters_own(sizes):
    systems = [ic.plummer(n, 11 + k) for k, n in enumerate(sizes)]
    with EnsembleHIP(systems, E2, precision="exact") as e:
        e.init()
        first = e.download()
        infos = e.run(1.0, 1.0, 6)
        last = e.download()
    for c in sorted({0, 1, 2, len(sizes) // 2, len(sizes) - 1}):
        r, v = systems[c]
        with Hermite4HIP(r, v, E2, precision="exact") as h:
            h.init_acc_jrk()
            a = h.init_dt()
            s = h.download()
            for q in first[c]:
                assert bits_equal(first[c][q], s[q]), (c, q)
            info, _, _ = h.run(0.0, a, 1.0, 1.0, 6)
            s = h.download()
            for q in last[c]:
                assert bits_equal(last[c][q], s[q]), (c, q)
            assert infos[c]["atime"] == info["atime"] and infos[c]["nsteps"] == info["nsteps"]
