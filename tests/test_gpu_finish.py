"""The block finish pass where its corrector changes form (32 and 33 active
particles of a block) and where the lanes per particle change (8, 32 and 128
j chunks): the corrector is the oracle's, bit for bit, on the forces the
step made."""
import numpy as np
import pytest

from gravidy_amd import Hermite4HIP

from test_gpu_parity import E2, bits_equal, block_state, check_forces

pytestmark = pytest.mark.gpu
T1 = 1.0 + 2.0 ** -12


@pytest.mark.parametrize("n", [1025, 2048, 8192, 8449, 33000])
@pytest.mark.parametrize("per_block", [1, 8, 9, 31, 32, 33, 256])
def test_finish_block_corrector_forms(oracle, n, per_block):
    r, v, f, t, dt = block_state(n, n + per_block, T1)
    rng = np.random.default_rng(n + per_block)
    dt[:] = 2.0 ** -rng.integers(3, 10, size=n).astype(float)
    t[:] = 1.0
    # per_block active particles in block 1, one in the last block
    mo = np.sort(np.append(256 + rng.choice(256, per_block, replace=False), n - 1)).astype(np.uint32)
    dt[mo] = 2.0 ** -12
    with Hermite4HIP(r, v, E2, precision="fp64") as h:
        h.upload(r, v, f, t, dt)
        k, atime = h.step(T1)
        s = h.download()
    assert k == mo.size
    po, pmo = oracle.predicted_pos_vel(T1, t, r, v, f)
    check_forces(s["f"], oracle.update_acc_jrk(mo, po, pmo, E2, f), mo, po, pmo, E2,
                 f"finish n={n} per_block={per_block}")
    z3 = np.zeros((n, 3))
    a2, a3, rc, vc, tc, dtc = oracle.correction_pos_vel(T1, mo, po, s["f"], f, z3, z3, r, v, t, dt)
    assert bits_equal(s["r"][:, :3], rc[:, :3]) and bits_equal(s["v"][:, :3], vc[:, :3])
    assert bits_equal(s["a2"][mo], a2[mo]) and bits_equal(s["a3"][mo], a3[mo])
    assert bits_equal(s["t"], tc) and bits_equal(s["dt"], dtc)
    assert atime == oracle.next_integration_time(tc, dtc)
