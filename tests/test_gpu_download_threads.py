"""h4h_download around 1 MB, from where two threads copy: the arrays as
uploaded, bit for bit."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP, ic

from test_gpu_download import check
from test_gpu_parity import E2

pytestmark = pytest.mark.gpu


# 28 doubles per particle, 4 of r alone: 131072 doubles are 1 MB
@pytest.mark.parametrize("n", [4681, 4682, 9362, 9363, 32767, 32768, 32769])
def test_one_and_two_threads(n):
    r, v = ic.plummer(n, n)
    f = np.random.default_rng(n).normal(size=(n, 6))
    with Hermite4HIP(r, v, E2) as h:
        h.upload(r, v, f, np.zeros(n), np.full(n, 2.0 ** -5))
        check(h, n, {"r": r, "f": f})
        h.step(2.0 ** -5)
        check(h, n, {})
