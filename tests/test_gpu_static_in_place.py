"""h4h_update_acc_jrk_static with the forces written over the particles it reads
(d_f6 on d_p6, or on d_pm): the rows of a call with arrays of their own."""
import numpy as np
import pytest
import torch

import gravidy_amd
from gravidy_amd import _lib, ic

from test_gpu_parity import E2, bits_equal

pytestmark = pytest.mark.gpu


def _call(p6, pm, n, move, f6, precision):
    lib = gravidy_amd.load()
    _lib.check("h4h_update_acc_jrk_static", lib.h4h_update_acc_jrk_static(
        p6.data_ptr(), pm.data_ptr(), n, move.data_ptr(), move.numel(), E2, precision,
        f6.data_ptr(), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return f6.cpu().numpy()


@pytest.mark.parametrize("precision", [gravidy_amd.H4H_FP64, gravidy_amd.H4H_MIXED,
                                       gravidy_amd.H4H_FP64_EXACT])
@pytest.mark.parametrize("n,nact", [(64, 3), (300, 24), (1024, 24), (1024, 100), (1000, 200),
                                    (1024, 256), (1024, 1024), (3000, 100)])
def test_in_place(n, nact, precision):
    r, v = ic.plummer(n, n + nact)
    dev = torch.device("cuda")
    rows = np.random.default_rng(nact).choice(n, nact, replace=False)
    move = torch.tensor(rows.astype(np.int32), device=dev)
    host = np.concatenate([r[:, :3], v[:, :3]], axis=1)
    mass = torch.tensor(r[:, 3].astype(np.float32), device=dev)
    p6 = torch.tensor(host, device=dev)
    own = _call(p6, mass, n, move, torch.zeros((n, 6), dtype=torch.float64, device=dev), precision)
    want = host.copy()
    want[rows] = own[rows]
    assert bits_equal(_call(p6, mass, n, move, p6, precision), want)
    # masses in the last rows of the forces
    f6 = torch.zeros((n, 6), dtype=torch.float64, device=dev)
    pm = f6.view(-1).view(torch.float32)[-n:]
    pm.copy_(mass)
    want = f6.cpu().numpy()
    want[rows] = own[rows]
    p6 = torch.tensor(host, device=dev)
    assert bits_equal(_call(p6, pm, n, move, f6, precision), want)
