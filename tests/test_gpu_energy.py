"""Energy sums at the edges of their work split (i blocks of 512, j chunks
of 16 to 256, workgroup counts) against the oracle, and a batch of clusters
against each cluster alone.  Tolerance: the energy's contract, 1e-13
relative."""
import numpy as np
import pytest

from gravidy_amd import EnsembleHIP, Hermite4HIP, ic, softening_e2

pytestmark = pytest.mark.gpu
E2 = softening_e2(1e-4)


@pytest.mark.parametrize("n", [1, 2, 16, 17, 511, 512, 513, 1023, 1025, 2049, 4097, 20001, 33000])
def test_energy_at_block_and_chunk_edges(oracle, n):
    r, v = ic.plummer(n, 900 + n) if n > 1 else (np.array([[1.0, 2.0, 3.0, 0.5]]),
                                                 np.array([[0.1, 0.2, 0.3, 0.0]]))
    with Hermite4HIP(r, v, E2) as h:
        ek, ep = h.get_energy()
    eko, epo = oracle.get_energy(r, v)
    assert abs(ek - eko) <= 1e-13 * abs(eko)
    assert abs(ep - epo) <= 1e-13 * abs(epo)


def test_energy_of_particles_coincident_across_chunks_is_minus_infinity():
    """Two particles at one position, in one i block and in two."""
    for n, a, b in ((1500, 3, 400), (1500, 3, 1400)):
        r, v = ic.plummer(n, 5)
        r[b, :3] = r[a, :3]
        with Hermite4HIP(r, v, E2) as h:
            ek, ep = h.get_energy()
        assert np.isfinite(ek) and ep == -np.inf


def test_ensemble_energies_equal_each_cluster_alone():
    sizes = [1, 3, 255, 256, 257, 600, 1024, 5000, 9001]
    systems = [ic.plummer(n, 40 + n) if n > 1 else (np.array([[0.0, 0.0, 0.0, 1.0]]),
                                                    np.zeros((1, 4))) for n in sizes]
    with EnsembleHIP(systems, E2) as ens:
        ek, ep = ens.energy()
    for c, (r, v) in enumerate(systems):
        with Hermite4HIP(r, v, E2) as h:
            assert h.get_energy() == (ek[c], ep[c])
