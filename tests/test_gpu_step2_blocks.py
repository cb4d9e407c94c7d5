"""The unsplit 2D step's workgroups (unsplit.hpp unsplit_block): four wavefronts march
one above the other and hand the first row's contributions down through local memory.
Heights around the shares of rows, bit for bit against the oracle's step2 (FP64, with
aux fields and a capacity too); in FP32 + Kahan the result does not depend on the shares
and stays within rounding of the oracle's."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests._cases import seeded_state

pytestmark = pytest.mark.gpu


SHAPES = [(61, 2), (7, 3), (64, 4), (130, 5), (60, 7), (59, 8), (3, 15), (121, 16), (62, 39),
          (20, 131)]


@pytest.mark.parametrize("rows", [None, 1, 5])
@pytest.mark.parametrize("mx,my", SHAPES)
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


# kind, meqn, transverse, capacity field, aux fields
@pytest.mark.parametrize("case", [(7, 1, 2, 2, 3), (8, 3, 2, 2, 3), (8, 3, 2, -1, 2), (6, 2, 0, 2, 3)])
@pytest.mark.parametrize("mx,my", SHAPES)
def test_unsplit_blocks_aux_capa_bit_exact(mx, my, case, monkeypatch):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    kind, meqn, trans, capa, maux = case
    ng, bcl, bcu = 2, [1, 2], [3, 2]
    print("unsplit blocks aux", (mx, my), case, flush=True)
    rng = np.random.default_rng(mx * my + kind)
    q = np.asfortranarray(rng.uniform(-1.0, 2.0, (meqn, mx, my)))
    aux = rng.uniform(-1.5, 1.5, (maux, mx, my))
    if kind == 8:      # density and sound speed
        aux[:2] = rng.uniform(0.5, 2.0, (2, mx, my))
    if capa >= 0:
        aux[capa] = rng.uniform(0.5, 2.0, (mx, my))
    aux = np.asfortranarray(aux)
    dx, dy = 1.0 / mx, 0.8 / my
    dt = 0.1 * min(dx, dy)
    meth = O.method_array(transverse=trans, num_aux=maux, index_capa=capa)
    qbc, abc = O.with_ghosts(q, ng), O.with_ghosts(aux, ng)
    O.bc2(qbc, ng, bcl, bcu)
    O.bc2(abc, ng, bcl, bcu, reflect=(-1, -1))
    ref = qbc.copy(order="F")
    lim = [4] * O.MWAVES[kind]
    c = O.step2(O.make_rp(kind, meqn=meqn), qbc, ref, ng, dx, dy, dt, meth, lim, aux=abc)
    qi = q_to_device(q)
    for rows in (None, 1, 3):
        if rows:
            monkeypatch.setenv("CLAWHIP_UNSPLIT_ROWS", str(rows))
        qo = torch.empty_like(qi)
        cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
        K.step2_unsplit(K.make_rp(kind, {}, meqn=meqn), qi, qo, cfl, bcl, bcu, [1, 2], meth, lim,
                        dx, dy, dt, aux=q_to_device(aux), aux_bc_lower=bcl, aux_bc_upper=bcu)
        torch.cuda.synchronize()
        assert np.array_equal(q_from_device(qo), O.interior(ref, ng)), rows
        assert float(cfl.item()) == c


@pytest.mark.parametrize("kind", [O.ACOUSTICS, O.EULER, O.SHALLOW, O.EULER5])
@pytest.mark.parametrize("mx,my", SHAPES)
def test_unsplit_blocks_fp32_whatever_the_shares(mx, my, kind, monkeypatch):
    """The compensation is of a few units in the last place; a cell's change is the sum of
    some 80 products of terms no larger than 4 max|q| times the Courant number c, each
    rounded to 2^-24."""
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    ng, bcl, bcu = 2, [1, 2], [3, 2]
    print("unsplit blocks fp32", (mx, my), kind, flush=True)
    rng = np.random.default_rng(mx * my + kind)
    q = seeded_state(rng, kind, (mx, my)).astype(np.float32).astype(np.float64)
    comp = (1e-7 * rng.standard_normal(q.shape)).astype(np.float32).astype(np.float64)
    meth, lim = O.method_array(transverse=2), [4] * O.MWAVES[kind]
    dx, dy = 1.0 / mx, 0.8 / my
    dt = 0.1 * min(dx, dy)
    qbc = O.with_ghosts(np.asfortranarray(q - comp), ng)
    O.bc2(qbc, ng, bcl, bcu)
    ref = qbc.copy(order="F")
    c = O.step2(O.make_rp(kind), qbc, ref, ng, dx, dy, dt, meth, lim)
    rp = K.make_rp(kind, {O.ACOUSTICS: dict(rho=1.0, bulk=4.0), O.SHALLOW: dict(grav=1.0)}.get(
        kind, dict(gamma=1.4)))
    qi, ci = q_to_device(np.asfortranarray(q), 1), q_to_device(np.asfortranarray(comp), 1)
    first = None
    for rows in (None, 1, 2, 5, 64):
        if rows:
            monkeypatch.setenv("CLAWHIP_UNSPLIT_ROWS", str(rows))
        qo, co = torch.empty_like(qi), torch.empty_like(ci)
        cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
        K.step2_unsplit(rp, qi, qo, cfl, bcl, bcu, [1, 2], meth, lim, dx, dy, dt, comp_in=ci,
                        comp_out=co)
        torch.cuda.synchronize()
        got = (q_from_device(qo), q_from_device(co), float(cfl.item()))
        if first is None:
            first = got
            out = got[0] - got[1]
            bound = 80 * 4 * c * 2.0 ** -24 * np.abs(q).max()
            assert np.abs(out - O.interior(ref, ng)).max() <= bound
            assert abs(got[2] - c) <= 50 * 2.0 ** -24 * c
        assert all(np.array_equal(a, b) for a, b in zip(got, first)), rows
