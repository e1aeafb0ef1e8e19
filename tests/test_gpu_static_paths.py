"""h4h_update_acc_jrk_static where its launches change: one launch (one j
chunk of up to four tiles, up to 256 active particles) and three; bit for bit
h4h_update_acc_jrk on a context, and an index out of range in the first and
last entries of the list."""
import numpy as np
import pytest

from gravidy_amd import softening_e2

from test_zz_no_alloc import SENTINEL, _check, _static, _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed", "exact"])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1024, 1025])
def test_static_paths_match_context(n, precision):
    r, v, p6, pm = _system(n, n + 1)
    rng = np.random.default_rng(n)
    for nact in (1, 4, 5, 16, 17, 48, 64, 128, 129, 191, 255, 256, 257, 1024):
        if nact <= n:
            move = rng.permutation(n)[:nact].astype(np.uint32)
            _check(r, v, p6, pm, move, softening_e2(1e-4), precision)


@pytest.mark.parametrize("n,nact", [(1000, 24), (1000, 128), (1000, 900), (5000, 1024), (5000, 1025),
                                    (65536, 40000)])
@pytest.mark.parametrize("at", [0, -1])
def test_static_paths_flag_bad_indices(n, nact, at):
    _, _, p6, pm = _system(n, 2)
    move = np.random.default_rng(n).permutation(n)[:nact].astype(np.uint32)
    good = move.copy()
    move[at] = n
    e2 = softening_e2(1e-4)
    f = _static(p6, pm, move, e2, "fp64")
    rest = np.ones(n, bool)
    rest[move[move < n]] = False
    assert np.isnan(f[~rest]).all() and (f[rest] == SENTINEL).all()
    f = _static(p6, pm, good, e2, "fp64")
    assert np.isfinite(f[good]).all()
