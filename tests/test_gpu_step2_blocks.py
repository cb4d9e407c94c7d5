"""The unsplit 2D step's workgroups (unsplit.hpp unsplit_block): four wavefronts march
one above the other and hand the first row's contributions down through local memory.
Heights around the shares of rows, bit for bit against the oracle's step2 (FP64)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests._cases import seeded_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [None, 1, 5])
@pytest.mark.parametrize("mx,my", [(61, 2), (7, 3), (64, 4), (130, 5), (60, 7), (59, 8), (3, 15),
                                   (121, 16), (62, 39), (20, 131)])
def test_unsplit_blocks_bit_exact(mx, my, rows, monkeypatch):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    if rows:
        monkeypatch.setenv("CLAWHIP_UNSPLIT_ROWS", str(rows))
    ng, bcl, bcu = 2, [1, 2], [1, 2]
    print("unsplit blocks", (mx, my, rows), flush=True)
    q = seeded_state(np.random.default_rng(mx * my), O.EULER, (mx, my))
    meth = O.method_array(transverse=2)
    dx, dy = 1.0 / mx, 0.8 / my
    dt = 0.2 * min(dx, dy)
    qbc = O.with_ghosts(q, ng)
    O.bc2(qbc, ng, bcl, bcu)
    ref = qbc.copy(order="F")
    c = O.step2(O.make_rp(O.EULER), qbc, ref, ng, dx, dy, dt, meth, [4] * 3)
    qi = q_to_device(q)
    qo = torch.empty_like(qi)
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    K.step2_unsplit(K.make_rp(2, {"gamma": 1.4}), qi, qo, cfl, bcl, bcu, [1, 2], meth, [4] * 3,
                    dx, dy, dt)
    torch.cuda.synchronize()
    assert np.array_equal(q_from_device(qo), O.interior(ref, ng))
    assert float(cfl.item()) == c
