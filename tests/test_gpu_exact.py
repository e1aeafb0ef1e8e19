"""The FP64_EXACT update at the edges of its work split: one or three active
particles per workgroup over j tiles of 192 or 64, and one lane per active
particle.  Every variant adds a particle's terms in ascending j, so each
result equals the oracle's bit for bit."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP, ic, softening_e2

pytestmark = pytest.mark.gpu


def _check(oracle, n, nact, e2, sample=None):
    r, v = ic.plummer(n, 31 + n)
    rng = np.random.default_rng(n + nact)
    move = np.sort(rng.choice(n, size=nact, replace=False)).astype(np.uint32)
    with Hermite4HIP(r, v, e2, precision="exact") as h:
        h.set_active(move)
        h.update_acc_jrk(nact)
        f = h.download()["f"]
    rows = move if sample is None else np.sort(rng.choice(move, size=sample, replace=False))
    p = np.concatenate([r[:, :3], v[:, :3]], axis=1)
    fo = oracle.update_acc_jrk(rows, p, r[:, 3].astype(np.float32), e2, np.zeros((n, 6)))
    assert f[rows].tobytes() == fo[rows].tobytes()
    idle = np.ones(n, bool)
    idle[move] = False
    assert not f[idle].any()


@pytest.mark.parametrize("n", [2, 63, 64, 65, 191, 192, 193, 256, 257, 385])
@pytest.mark.parametrize("softened", [True, False])
def test_exact_update_j_tile_edges(oracle, n, softened):
    for nact in {1, n // 2, n}:
        _check(oracle, n, nact, softening_e2(1e-4) if softened else 0.0)


@pytest.mark.parametrize("nact", [768, 769, 770, 771, 1537])
def test_exact_update_items_of_one_and_three(oracle, nact):
    _check(oracle, 1537, nact, softening_e2(1e-4))


@pytest.mark.parametrize("nact", [45055, 45056, 45099])
def test_exact_update_one_lane_per_particle(oracle, nact):
    _check(oracle, 45099, nact, softening_e2(1e-4), sample=200)
