"""The unsplit 3D step lays its slices end to end over the wavefronts
(unsplit3.hip k_flux3): slice lengths around a wavefront's 60 owned cells and far
below them, one slice ending anywhere in a wavefront, in each direction, bit for
bit against the oracle and within the work array; a step onto its own input, which the
directions would read back half done, is refused."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests._cases import seeded_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 2, 2), (3, 2, 5), (56, 3, 2), (2, 57, 3), (3, 2, 60),
                                   (61, 2, 64), (5, 116, 2), (121, 4, 3)])
def test_step3_slices_bit_exact(shape):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    print("step3 slices", shape, flush=True)
    q = seeded_state(np.random.default_rng(sum(shape)), O.EULER3, shape)
    ng, bcl, bcu = 2, [1, 3, 2], [1, 3, 2]
    dx, dy, dz = 1.0 / shape[0], 0.9 / shape[1], 1.1 / shape[2]
    dt = 0.1 * min(dx, dy, dz)
    meth = [1, 2, 22, 0, 0, 0, 0]
    qbc = O.with_ghosts(q, ng)
    O.bc3(qbc, ng, bcl, bcu)
    ref = qbc.copy(order="F")
    c_ref = O.step3(O.make_rp(O.EULER3), qbc, ref, ng, dx, dy, dz, dt, meth, [4] * 3)
    rp = K.make_rp(5, {"gamma": 1.4})
    qi = q_to_device(q)
    out = torch.empty_like(qi)
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    n = int(K.L.lib().clawhip_step3_unsplit_work_elems(5, *shape))
    work = torch.full((n + 512,), -1.5, dtype=torch.float64, device="cuda")
    K.step3_unsplit(rp, qi, out, cfl, bcl, bcu, [1, 2, 3], meth, [4] * 3, dx, dy, dz, dt,
                    work=work[:n])
    torch.cuda.synchronize()
    assert bool((work[n:] == -1.5).all())
    assert np.array_equal(q_from_device(out), O.interior(ref, ng))
    assert float(cfl.item()) == c_ref


def test_step3_onto_its_input_is_refused():
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_to_device
    qi = q_to_device(seeded_state(np.random.default_rng(1), O.EULER3, (4, 5, 6)))
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    with pytest.raises(K.L.ClawhipError):
        K.step3_unsplit(K.make_rp(5, {"gamma": 1.4}), qi, qi, cfl, [1] * 3, [1] * 3, [1, 2, 3],
                        [1, 2, 22, 0, 0, 0, 0], [4] * 3, 0.25, 0.2, 0.2, 0.01)
