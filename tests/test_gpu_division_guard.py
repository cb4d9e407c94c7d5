"""Where the FP64 solves' shared reciprocals give way to the plain division
(riemann.hpp Watch, march_both): products of two small values among the numerators,
states that are small as a whole, a march that meets the first value out of bounds in
any of its rows, parameters out of range.  Bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests._cases import seeded_state

pytestmark = pytest.mark.gpu

SOLVERS = [O.SHALLOW, O.SHALLOW_HLLE, O.EULER, O.EULER5]


def _classic2(kind, q, split=False, grav=1.0, dt_scale=0.1):
    """One classic step on the device and by the oracle."""
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    mx, my, ng, bc = q.shape[1], q.shape[2], 2, [1, 1]
    dx, dy = 1.0 / mx, 0.9 / my
    dt, lim = dt_scale * min(dx, dy), [4] * O.MWAVES[kind]
    qbc = O.with_ghosts(q, ng)
    O.bc2(qbc, ng, bc, bc)
    rp = O.make_rp(kind, gamma=1.4, grav=grav)
    ref = qbc.copy(order="F")
    meth = O.method_array(dimensional_split=True) if split else \
        O.method_array(transverse=0 if kind == O.SHALLOW_HLLE else 2)
    if split:
        c = max(O.step2(rp, qbc, ref, ng, dx, dy, dt, meth, lim, ids=1),
                O.step2(rp, ref.copy(order="F"), ref, ng, dx, dy, dt, meth, lim, ids=2))
    else:
        c = O.step2(rp, qbc, ref, ng, dx, dy, dt, meth, lim)
    qi = q_to_device(q)
    qo = torch.empty_like(qi)
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    (K.step2_split if split else K.step2_unsplit)(
        K.make_rp(kind, {"gamma": 1.4, "grav": grav}), qi, qo, cfl, bc, bc, [1, 2], meth, lim, dx,
        dy, dt)
    torch.cuda.synchronize()
    return q_from_device(qo), float(cfl.item()), O.interior(ref, ng), c


def _sharp2(kind, q, cd, grav=1.0, dt_scale=0.1):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    mx, my, ng, bc = q.shape[1], q.shape[2], 3, [1, 1]
    qbc = O.with_ghosts(q, ng)
    O.bc2(qbc, ng, bc, bc)
    dx, dy = 1.0 / mx, 0.9 / my
    dt = dt_scale * min(dx, dy)
    dq, c = O.sharp_flux2(O.make_rp(kind, gamma=1.4, grav=grav), qbc, ng, dx, dy, dt, cd)
    qi = q_to_device(q)
    out = torch.empty_like(qi)
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    K.sharp2_stage(K.make_rp(kind, {"gamma": 1.4, "grav": grav}), cd, out, cfl, bc, bc, [1, 2],
                   dt, dx, dy, qi)
    torch.cuda.synchronize()
    return q_from_device(out), float(cfl.item()), O.interior(dq, ng), c


def _equal(result):
    got, cfl, ref, c = result
    assert np.array_equal(got, ref, equal_nan=True), np.argwhere(~(got == ref))[:4]
    assert cfl == c


def _shear(kind, shape, exponents, rho, rng):
    """A uniform gas or depth rho with a transverse momentum alone, of the magnitudes
    10^exponents: the other momentum changes by products of two such values only."""
    q = np.zeros((O.MEQN[kind],) + shape)
    tiny = np.sign(rng.uniform(-1, 1, shape)) * 10.0 ** rng.uniform(*exponents, shape)
    q[0] = rho
    q[2] = tiny
    if kind == O.EULER3:
        q[2], q[3] = 0.0, tiny
    if kind not in (O.SHALLOW, O.SHALLOW_HLLE):
        q[3 + (kind == O.EULER3)] = 0.9 * rho   # 2 a = 1.42
    if kind == O.EULER5:
        q[4] = rng.uniform(0, 1, shape)
    return np.asfortranarray(q)


# squares around the smallest numbers, around 2^-960, around 2^-800 and above
@pytest.mark.parametrize("exponents", [(-162.5, -152.0), (-155.0, -142.0), (-125.0, -117.0),
                                       (-115.0, -94.0)])
@pytest.mark.parametrize("rho", [1.0, 1.37])
@pytest.mark.parametrize("kind", SOLVERS)
def test_products_of_small_values(kind, rho, exponents):
    print("guard products", kind, rho, exponents, flush=True)
    q = _shear(kind, (130, 23), exponents, rho, np.random.default_rng(kind))
    for split in (False, True):
        _equal(_classic2(kind, q, split))
    if kind != O.EULER5:
        for cd in (0, 2):
            _equal(_sharp2(kind, q, cd))


@pytest.mark.parametrize("power", [-98, -101, -320, -505, -520])
@pytest.mark.parametrize("kind", SOLVERS)
def test_all_fields_small(kind, power):
    """A state scaled to about 2^power: squares of its momenta over its densities are of its
    energies' size."""
    q = np.asfortranarray(2.0 ** power * seeded_state(np.random.default_rng(kind), kind, (66, 23)))
    grav = 2.0 ** min(-power, 55)
    for split in (False, True):
        _equal(_classic2(kind, q, split, grav, 0.05))
    if kind != O.EULER5:
        _equal(_sharp2(kind, q, 0, grav, 0.05))


@pytest.mark.parametrize("exponents", [(-162.5, -152.0), (-155.0, -142.0), (-125.0, -117.0)])
def test_products_of_small_values_3d(exponents):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    n, ng, bc = (66, 9, 7), 2, [1, 1, 1]
    q = _shear(O.EULER3, n, exponents, 1.37, np.random.default_rng(3))
    d = [1.0 / n[0], 0.9 / n[1], 1.1 / n[2]]
    dt, lim, rp = 0.1 * min(d), [4] * 3, O.make_rp(O.EULER3)
    qbc = O.with_ghosts(q, ng)
    O.bc3(qbc, ng, bc, bc)
    for split in (False, True):
        meth = O.method_array(dimensional_split=True) if split else [1, 2, 22, 0, 0, 0, 0]
        ref = qbc.copy(order="F")
        if split:
            c = max(O.step3ds(rp, src, ref, ng, *d, dt, meth, lim, k)
                    for k, src in ((1, qbc), (2, ref), (3, ref)))
        else:
            c = O.step3(rp, qbc, ref, ng, *d, dt, meth, lim)
        qi = q_to_device(q)
        qo = torch.empty_like(qi)
        cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
        (K.step3_split if split else K.step3_unsplit)(K.make_rp(5, {"gamma": 1.4}), qi, qo, cfl,
                                                      bc, bc, [1, 2, 3], meth, lim, *d, dt)
        torch.cuda.synchronize()
        _equal((q_from_device(qo), float(cfl.item()), O.interior(ref, ng), c))


@pytest.mark.parametrize("scale", [1.0, 2.0 ** 39, 2.0 ** 60, 2.0 ** 80])
@pytest.mark.parametrize("kind", [O.SHALLOW, O.SHALLOW_HLLE, O.EULER])
def test_small_edge_values_beside_a_zero_region(kind, scale):
    """WENO5 gives a zero region beside jumps edge values of eps^2 / jump^3."""
    rng = np.random.default_rng(kind)
    q = _shear(kind, (66, 23), (-2.0, -0.5), 1.37, rng)
    q[2, :, :] *= rng.uniform(0, 1, (66, 23)) < 0.15
    q = np.asfortranarray(scale * q)
    for cd in (0, 2):
        _equal(_sharp2(kind, q, cd, 1.0 / scale))


def _one_row(kind, shape, row, what, rng):
    """An ordinary state but for one row, in half of the columns: its momenta below their
    lower bound (2^-800 = 1.5e-241), around it, around the Euler solvers' (2^-320 =
    4.7e-97) or near the smallest numbers; its cells scaled beyond the upper bound
    (2^100), around it, around the Euler solvers' (2^40), or around the lower bound of
    densities, depths and energies (2^-100)."""
    q = seeded_state(rng, kind, shape)
    if kind in (O.EULER, O.EULER5):   # milder noise keeps edge pressures positive
        mean = seeded_state(np.random.default_rng(0), kind, (1, 1)).mean(axis=(1, 2))
        q = np.asfortranarray(0.85 * mean[:, None, None] + 0.15 * q)
    at = slice(0, shape[0] // 2)
    powers = {"large": 205, "upper": 100, "middle": 40, "thin": -100}
    if what in powers:
        q[:, at, row] *= 2.0 ** powers[what]
    else:
        size = {"small": 1e-250, "denormal": 1e-315,
                "lower": 10.0 ** rng.uniform(-243.0, -239.0, q[1:3, at, row].shape),
                "narrow": 10.0 ** rng.uniform(-98.0, -94.0, q[1:3, at, row].shape)}[what]
        q[1:3, at, row] *= size
    return q


@pytest.mark.parametrize("what", ["small", "lower", "narrow", "denormal", "large", "upper",
                                  "middle", "thin"])
@pytest.mark.parametrize("kind", SOLVERS)
def test_first_such_row_anywhere_in_a_march(kind, what, monkeypatch):
    """Four wavefronts of nine rows each (one block of 35), and marches of nine rows in the
    split sweeps and the SharpClaw stages: the row at every place in them, that of the rows
    handed from one wavefront to the next among them."""
    for name in ("UNSPLIT", "SPLIT", "SHARP"):
        monkeypatch.setenv("CLAWHIP_%s_ROWS" % name, "9")
    rng = np.random.default_rng(kind + len(what))
    for row in range(35):
        print("guard row", kind, what, row, flush=True)
        q = _one_row(kind, (66, 35), row, what, rng)
        for split in (False, True):
            _equal(_classic2(kind, q, split, dt_scale=0.01))
        if kind != O.EULER5:
            _equal(_sharp2(kind, q, 2 * (row % 2), dt_scale=0.01))


@pytest.mark.parametrize("grav", [2.0 ** -300, 2.0 ** -62, 2.0 ** 62, 2.0 ** 300])
@pytest.mark.parametrize("kind", [O.SHALLOW, O.SHALLOW_HLLE])
def test_parameters_out_of_range(kind, grav):
    q = seeded_state(np.random.default_rng(kind), kind, (66, 21))
    scale = 0.1 / max(1.0, grav) ** 0.5
    for split in (False, True):
        _equal(_classic2(kind, q, split, grav, scale))
    for cd in (0, 2):
        _equal(_sharp2(kind, q, cd, grav, scale))
