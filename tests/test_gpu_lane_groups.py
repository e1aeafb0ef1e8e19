"""Steps of more than 128 active particles whose work items would be few: the
plan takes narrower lane groups than the active count alone would give.  At
the lines of that rule, FP64 forces against the oracle's and mixed forces
against 256-slot groups, whose FP32 runs the narrower ones keep."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP, ic

from test_gpu_parity import E2, check_forces, p6, pm_of, term_scales

pytestmark = pytest.mark.gpu

# (n, nact): one and four j tiles, the first narrowed count, full and ragged
# last groups, the last narrowed and first wide ones (n_it tiles below 1024 at
# 256 slots; below 512 at 64)
CASES = [(200, 129), (256, 256), (1000, 129), (1024, 1023), (1025, 145), (4096, 1985), (4096, 2048),
         (4096, 4096), (10007, 768), (10007, 769), (10007, 6400), (10007, 6401), (70000, 200)]


def forces(r, v, n, move, precision, tuning=None):
    with Hermite4HIP(r, v, E2, precision=precision) as h:
        if tuning is not None:
            h.set_tuning(tuning)
        h.set_active(move)
        h.update_acc_jrk(move.size)
        return h.download()["f"]


def system(n, nact):
    r, v = ic.plummer(n, n + nact)
    move = np.sort(np.random.default_rng(n + nact).choice(n, nact, replace=False)).astype(np.uint32)
    return r, v, move


@pytest.mark.parametrize("n,nact", CASES)
def test_narrow_groups_fp64(oracle, n, nact):
    r, v, move = system(n, nact)
    idx = move if n * nact < 5e6 else move[:: n * nact // 5_000_000 + 1]
    p, pm = p6(r, v), pm_of(r)
    fo = oracle.update_acc_jrk(idx, p, pm, E2, np.zeros((n, 6)))
    check_forces(forces(r, v, n, move, "fp64"), fo, idx, p, pm, E2, f"groups n={n} nact={nact}")


@pytest.mark.parametrize("n,nact", [(a, b) for a, b in CASES if b >= 192])
def test_narrow_groups_mixed_keep_their_runs(n, nact):
    r, v, move = system(n, nact)
    narrow = forces(r, v, n, move, "mixed")
    wide = forces(r, v, n, move, "mixed", {int(np.log2(nact)): (0, 256)})
    # two orders of the same n / 32 run sums in FP64, each within runs 2^-53
    # of the sum of their magnitudes
    tol = 2.0 * (n / 32 + 1) * 2.0 ** -53 * 1.001
    p, pm = p6(r, v), pm_of(r)
    for i in move[:: max(1, nact // 64)]:
        sa, sj = term_scales(int(i), p, pm, E2)
        d = narrow[i] - wide[i]
        assert np.linalg.norm(d[:3]) <= tol * sa and np.linalg.norm(d[3:]) <= tol * sj
