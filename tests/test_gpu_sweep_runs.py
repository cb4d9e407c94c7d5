"""The y and z sweeps of the dimension-split steps cut a pencil into runs of rows
(classic_split.hip k_march): in place, four runs to a workgroup, each reading its
neighbours' rows before they are rewritten; out of place, runs sized to fill the
device.  Lengths around the runs' edges, bit for bit against the oracle's
step2ds / step3ds (FP64)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests._cases import seeded_state

pytestmark = pytest.mark.gpu


EXTRAP = ([1, 1, 1], [1, 1, 1])
SIDES3 = [([2, 2, 2], [2, 2, 2]), ([3, 3, 3], [3, 3, 3]), ([1, 3, 2], [3, 1, 2]),
          ([2, 1, 3], [2, 3, 1])]


@pytest.mark.parametrize("my,sides", [(my, EXTRAP) for my in (2, 3, 4, 5, 7, 8, 9, 16, 17, 33)]
                         + [(my, s) for my in (2, 5, 8, 17) for s in SIDES3])
def test_split3_runs_bit_exact(my, sides):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    mx, mz, ng = 67, my + 2, 2
    print("split3 runs", (mx, my, mz), flush=True)
    bcl, bcu = sides
    q = seeded_state(np.random.default_rng(my), O.EULER3, (mx, my, mz))
    meth = O.method_array(dimensional_split=True)
    dx, dy, dz = 1.0 / mx, 0.9 / my, 1.1 / mz
    dt = 0.2 * min(dx, dy, dz)
    qbc = O.with_ghosts(q, ng)
    O.bc3(qbc, ng, bcl, bcu)
    qold = qbc.copy(order="F")
    rp = O.make_rp(O.EULER3)
    cs = [O.step3ds(rp, src, qbc, ng, dx, dy, dz, dt, meth, [4] * 3, k)
          for k, src in ((1, qold), (2, qbc), (3, qbc))]
    qi = q_to_device(q)
    qo = torch.empty_like(qi)
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    K.step3_split(K.make_rp(5, {"gamma": 1.4}), qi, qo, cfl, bcl, bcu, [1, 2, 3], meth, [4] * 3,
                  dx, dy, dz, dt)
    torch.cuda.synchronize()
    assert np.array_equal(q_from_device(qo), O.interior(qbc, ng))
    assert float(cfl.item()) == max(cs)


@pytest.mark.parametrize("sides", [([1, 1], [1, 1]), ([2, 3], [2, 1])])
@pytest.mark.parametrize("mx,my", [(3, 2), (64, 2), (61, 3), (200, 37), (5, 130), (130, 1030)])
def test_split2_runs_bit_exact(mx, my, sides):
    """Both forms of the 2D y sweep: out of place, and in place on a whole qbc."""
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    ng, (bcl, bcu) = 2, sides
    print("split2 runs", (mx, my), flush=True)
    q = seeded_state(np.random.default_rng(mx + my), O.SHALLOW, (mx, my))
    meth = O.method_array(dimensional_split=True)
    dx, dy = 1.0 / mx, 0.8 / my
    dt = 0.2 * min(dx, dy)
    qbc = O.with_ghosts(q, ng)
    O.bc2(qbc, ng, bcl, bcu)
    start = qbc.copy(order="F")
    ref = qbc.copy(order="F")
    rp = O.make_rp(O.SHALLOW)
    c = max(O.step2(rp, qbc, ref, ng, dx, dy, dt, meth, [4] * 3, ids=1),
            O.step2(rp, ref.copy(order="F"), ref, ng, dx, dy, dt, meth, [4] * 3, ids=2))
    krp = K.make_rp(3, {"grav": 1.0})
    for whole in (False, True):
        qi = q_to_device(start if whole else q)
        qo = torch.empty_like(qi)
        cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
        codes = ([4, 4], [4, 4]) if whole else (bcl, bcu)
        K.step2_split(krp, qi, qo, cfl, *codes, [1, 2], meth, [4] * 3, dx, dy, dt, whole=whole)
        torch.cuda.synchronize()
        out = q_from_device(qo)
        assert np.array_equal(O.interior(out, ng) if whole else out, O.interior(ref, ng))
        assert float(cfl.item()) == c


@pytest.mark.parametrize("mx,my,mz", [(60, 2, 3), (61, 3, 2), (59, 4, 5), (121, 9, 2), (2, 37, 4),
                                      (7, 130, 3), (64, 64, 5)])
def test_split3_fp32_one_pass_xy(mx, my, mz):
    """The FP32 + Kahan step's x- and y-sweep in one pass, against the FP64 oracle's three
    sweeps from the same FP32 state, with a compensation of a few units in the last place.
    A cell's change is three sums of some 50 products of terms no larger than 4 max|q|
    times the Courant number c, each rounded to 2^-24: 3 * 50 * 4 * c * 2^-24 max|q|."""
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    ng, bcl, bcu = 2, [1, 2, 3], [1, 2, 3]
    print("split3 xy", (mx, my, mz), flush=True)
    rng = np.random.default_rng(mx + my)
    q = seeded_state(rng, O.EULER3, (mx, my, mz)).astype(np.float32)
    comp = (1e-7 * rng.standard_normal(q.shape)).astype(np.float32)
    meth = O.method_array(dimensional_split=True)
    dx, dy, dz = 1.0 / mx, 0.9 / my, 1.1 / mz
    dt = 0.05 * min(dx, dy, dz)
    start = np.asfortranarray(q.astype(np.float64) - comp.astype(np.float64))
    qbc = O.with_ghosts(start, ng)
    O.bc3(qbc, ng, bcl, bcu)
    rp = O.make_rp(O.EULER3)
    cs = []
    for k in (1, 2, 3):
        src = qbc.copy(order="F") if k == 1 else qbc
        cs.append(O.step3ds(rp, src, qbc, ng, dx, dy, dz, dt, meth, [4] * 3, k))
    qi = q_to_device(np.asfortranarray(q.astype(np.float64))).float()
    ci = q_to_device(np.asfortranarray(comp.astype(np.float64))).float()
    qo, co = torch.empty_like(qi), torch.empty_like(ci)
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    K.step3_split(K.make_rp(5, {"gamma": 1.4}), qi, qo, cfl, bcl, bcu, [1, 2, 3], meth, [4] * 3,
                  dx, dy, dz, dt, comp_in=ci, comp_out=co)
    torch.cuda.synchronize()
    out = q_from_device(qo.double()) - q_from_device(co.double())
    bound = 3 * 50 * 4 * max(cs) * 2.0 ** -24 * np.abs(start).max()
    assert np.abs(out - O.interior(qbc, ng)).max() <= bound
    assert abs(float(cfl.item()) - max(cs)) <= 50 * 2.0 ** -24 * max(cs)


@pytest.mark.parametrize("sides", [EXTRAP] + SIDES3)
@pytest.mark.parametrize("mx,my,mz", [(60, 2, 3), (61, 3, 2), (121, 9, 5), (2, 37, 4), (7, 130, 3)])
def test_split3_fp32_carries_the_compensation(mx, my, mz, sides):
    """With dt = 0 the three sweeps of the FP32 + Kahan step change nothing, so the state
    less its compensation (varying from cell to cell, far above the rounding of the
    steps) comes out as it went in: each sweep adds -comp to q and keeps what the sum
    lost, exactly where |q| >= |comp|, within half a unit of comp elsewhere."""
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    print("split3 compensation", (mx, my, mz), sides, flush=True)
    rng = np.random.default_rng(mx + my + mz)
    q = seeded_state(rng, O.EULER3, (mx, my, mz)).astype(np.float32)
    comp = rng.uniform(-1e-3, 1e-3, q.shape).astype(np.float32)
    qi = q_to_device(np.asfortranarray(q.astype(np.float64)), 1)
    ci = q_to_device(np.asfortranarray(comp.astype(np.float64)), 1)
    qo, co = torch.empty_like(qi), torch.empty_like(ci)
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    K.step3_split(K.make_rp(5, {"gamma": 1.4}), qi, qo, cfl, *sides, [1, 2, 3],
                  O.method_array(dimensional_split=True), [4] * 3, 0.1, 0.1, 0.1, 0.0,
                  comp_in=ci, comp_out=co)
    torch.cuda.synchronize()
    out = q_from_device(qo.double()) - q_from_device(co.double())
    before = q.astype(np.float64) - comp.astype(np.float64)
    assert np.abs(out - before).max() <= 3 * 2.0 ** -24 * np.abs(comp).max()
