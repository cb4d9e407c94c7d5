"""The reference-equal FP64 solves share reciprocals between quotients while a
wavefront's values lie within bounds, and divide plainly otherwise (riemann.hpp
Divided, Watch).  States whose tails decay through the lower bound of momenta, 2^-800,
to denormals and zeros, in half of the columns of every row, are stepped bit for bit
as the oracle does, by every march that chooses (the choice in mid-march and the upper
bound: test_gpu_division_guard.py).  Acoustics divides plainly whatever the values."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests._cases import seeded_state
from tests.test_gpu_sharp import PD, _orp

pytestmark = pytest.mark.gpu

# decimal exponents of the values' magnitudes: around 2^-800 (1.5e-241), around 2^-700,
# down to the smallest denormal, around 2^200 (the linear solver only)
RANGES = {"bound": (-243.0, -239.0), "edge": (-213.0, -209.0), "denormal": (-323.5, -190.0),
          "large": (59.0, 61.5)}


def _tails(kind, shape, span, rng):
    """A state whose momenta (acoustics: every field) are of the span's magnitudes
    in about half of the columns, zero in some cells and ordinary elsewhere."""
    q = seeded_state(rng, kind, shape)
    tiny = np.sign(rng.uniform(-1, 1, q.shape)) * 10.0 ** rng.uniform(*RANGES[span], q.shape)
    tiny[rng.uniform(0, 1, q.shape) < 0.2] = 0.0
    at = slice(0, shape[0] // 2)
    if kind == O.ACOUSTICS:
        q[:, at] = tiny[:, at]
        return q
    nd = len(shape)
    q[0, at] = 1.0                     # at rest but for the tails
    q[1:1 + nd, at] = tiny[1:1 + nd, at]
    if kind != O.SHALLOW:
        q[nd + 1, at] = 2.5
    return q


CASES = [(O.ACOUSTICS, "edge"), (O.ACOUSTICS, "denormal"), (O.ACOUSTICS, "large"),
         (O.SHALLOW, "edge"), (O.SHALLOW, "denormal"), (O.EULER, "edge"), (O.EULER, "denormal"),
         (O.SHALLOW, "bound"), (O.EULER, "bound")]


def _device(q):
    from pyclaw_amd.device import q_to_device
    qi = q_to_device(q)
    return qi, torch.empty_like(qi), torch.zeros(1, dtype=torch.float64, device="cuda")


@pytest.mark.parametrize("kind,span", CASES)
def test_2d_steps_bit_exact(kind, span):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device
    rng = np.random.default_rng(10 * kind + len(span))
    mx, my, ng, bc = 130, 23, 2, [1, 1]
    q = _tails(kind, (mx, my), span, rng)
    dx, dy = 1.0 / mx, 0.9 / my
    dt, lim = 0.1 * dx, [4] * O.MWAVES[kind]
    qbc = O.with_ghosts(q, ng)
    O.bc2(qbc, ng, bc, bc)
    rp = K.make_rp(kind, PD[kind])
    for split in (False, True):
        meth = O.method_array(transverse=2, dimensional_split=split)
        ref = qbc.copy(order="F")
        if split:
            c = max(O.step2(_orp(kind), qbc, ref, ng, dx, dy, dt, meth, lim, ids=1),
                    O.step2(_orp(kind), ref.copy(order="F"), ref, ng, dx, dy, dt, meth, lim, ids=2))
        else:
            c = O.step2(_orp(kind), qbc, ref, ng, dx, dy, dt, meth, lim)
        qi, qo, cfl = _device(q)
        (K.step2_split if split else K.step2_unsplit)(rp, qi, qo, cfl, bc, bc, [1, 2], meth, lim,
                                                      dx, dy, dt)
        torch.cuda.synchronize()
        assert np.array_equal(q_from_device(qo), O.interior(ref, ng)), split
        assert float(cfl.item()) == c


@pytest.mark.parametrize("kind,span", CASES[:2] + CASES[3:])
def test_sharp_operator_bit_exact(kind, span):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device
    rng = np.random.default_rng(20 * kind + len(span))
    mx, my, ng, bc = 118, 23, 3, [2, 2]
    q = _tails(kind, (mx, my), span, rng)
    if kind == O.EULER:   # milder noise keeps WENO5's edge pressures positive
        q[:, mx // 2:] = 0.85 * np.array([1.0, 0.0, 0.0, 2.5])[:, None, None] \
            + 0.15 * q[:, mx // 2:]
    qbc = O.with_ghosts(q, ng)
    O.bc2(qbc, ng, bc, bc)
    dx, dy = 1.0 / mx, 0.9 / my
    dt = 0.1 * dx
    for cd in (0,) if kind == O.ACOUSTICS else (0, 2):
        dq, c = O.sharp_flux2(_orp(kind), qbc, ng, dx, dy, dt, cd)
        qi, out, cfl = _device(q)
        K.sharp2_stage(K.make_rp(kind, PD[kind]), cd, out, cfl, bc, bc, [1, 2], dt, dx, dy, qi)
        torch.cuda.synchronize()
        assert np.array_equal(q_from_device(out), O.interior(dq, ng), equal_nan=True), cd
        assert float(cfl.item()) == c


@pytest.mark.parametrize("span", ["edge", "denormal", "bound"])
def test_3d_steps_bit_exact(span):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device
    rng = np.random.default_rng(len(span))
    n, ng, bc = (66, 9, 7), 2, [1, 1, 1]
    q = _tails(O.EULER3, n, span, rng)
    d = [1.0 / n[0], 0.9 / n[1], 1.1 / n[2]]
    dt, lim, rp = 0.1 * min(d), [4] * 3, O.make_rp(O.EULER3)
    qbc = O.with_ghosts(q, ng)
    O.bc3(qbc, ng, bc, bc)
    krp = K.make_rp(5, {"gamma": 1.4})
    for split in (False, True):
        meth = O.method_array(dimensional_split=True) if split else [1, 2, 22, 0, 0, 0, 0]
        ref = qbc.copy(order="F")
        if split:
            c = max(O.step3ds(rp, src, ref, ng, *d, dt, meth, lim, k)
                    for k, src in ((1, qbc), (2, ref), (3, ref)))
        else:
            c = O.step3(rp, qbc, ref, ng, *d, dt, meth, lim)
        qi, qo, cfl = _device(q)
        (K.step3_split if split else K.step3_unsplit)(krp, qi, qo, cfl, bc, bc, [1, 2, 3], meth,
                                                      lim, *d, dt)
        torch.cuda.synchronize()
        assert np.array_equal(q_from_device(qo), O.interior(ref, ng)), split
        assert float(cfl.item()) == c
