"""Timed h4h_step calls: the update passes counted and timed are those of steps
that launch the update kernel; steps that one kernel makes by itself count in
the steps' time only."""
import pytest

from gravidy_amd import Hermite4HIP, ic

from test_gpu_parity import E2

pytestmark = pytest.mark.gpu


def _steps(h, r, v, count):
    h.upload(r, v)
    h.init_acc_jrk()
    a = h.init_dt()
    h.set_timing(True)
    h.stats(reset=True)
    sizes = []
    for _ in range(count):
        k, a = h.step(a)
        sizes.append(k)
    return sizes, h.stats()


@pytest.mark.parametrize("n,largest", [(300, 64), (1024, 64), (3000, 128), (20000, 128),
                                       (40000, 128), (70000, 0)])
def test_update_passes_of_steps(n, largest):
    """largest: the most active particles of a step in one launch."""
    r, v = ic.plummer(n, 5 * n)
    with Hermite4HIP(r, v, E2) as h:
        _steps(h, r, v, 40)  # (first launches)
        for _ in range(6):
            sizes, st = _steps(h, r, v, 120)
            assert st["block_steps"] == 120
            assert st["update_launches"] >= sum(k > largest for k in sizes)
            # (workgroups that do not come together leave their step to the launches)
            if st["update_launches"] == sum(k > largest for k in sizes):
                break
        assert st["update_launches"] == sum(k > largest for k in sizes)
        assert 0 < st["update_launches"]
        assert (largest == 0) or st["update_launches"] < 120
        assert st["small_steps"] == (sum(k <= largest for k in sizes) if n <= 1024 else 0)
        assert 0.0 < st["update_ms"] < st["step_ms"]
        # every pass counted ran the pairs: 1e12 a second at the very most
        pairs = sum(k * n for k in sizes if k > largest)
        assert st["update_ms"] * 1e-3 > pairs / 1.5e12
