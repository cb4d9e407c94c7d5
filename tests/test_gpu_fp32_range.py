"""FP32 + Kahan steps of states near the top of the FP32 range: wave norms between 2^63
and 2^64, whose squares (the limiter's denominators) lie between 2^126 and 2^128, and
WENO5 weights whose denominators do.  The equations are homogeneous (shallow water with
g scaled inversely), so a state scaled by 2^63 has 2^63 times the step of the state
itself: a limiter that took such a ratio as 0 would fall back to first order."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

S = 2.0 ** 63


def _contact(kind, shape, rng):
    """A state whose waves are of norms up to 1.6: one linearly degenerate family (plus
    rounding in the others), or for acoustics both."""
    if kind == O.ACOUSTICS:   # norm^2 = 5 a^2, |a| <= (1 + 2) * 0.9 / 4
        return rng.uniform(-0.45, 0.45, (3,) + shape)
    if kind == O.SHALLOW:     # a jump of h v alone
        return np.stack([np.full(shape, 1.5), np.full(shape, 0.3),
                         np.where(np.arange(shape[0])[:, None] % 7 < 3, 0.75, -0.5)
                         * rng.uniform(0.8, 1.0, shape)])
    nd = len(shape)           # a jump of density at rest pressure, uniform velocity
    rho = rng.uniform(1.0, 2.4, shape)
    vel = [0.25, -0.125, 0.0625][:nd]
    return np.stack([rho] + [rho * v for v in vel]
                    + [2.5 + 0.5 * rho * sum(v * v for v in vel)])


def _step(kind, q, scale, lim, form):
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    n = q.shape[1:]
    d = [1.0 / m for m in n]
    dt = 0.1 * min(d)
    rp = K.make_rp(kind, {O.ACOUSTICS: dict(rho=1.0, bulk=4.0),
                          O.SHALLOW: dict(grav=1.0 / scale)}.get(kind, dict(gamma=1.4)))
    qi = q_to_device(np.asfortranarray(scale * q), 1)
    assert torch.isfinite(qi).all()
    ci = torch.zeros_like(qi)
    qo, co = torch.empty_like(qi), torch.empty_like(qi)
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    bc = [1, 2, 3][:len(n)]
    lims = [lim] * O.MWAVES[kind]
    kw = dict(comp_in=ci, comp_out=co)
    if len(n) == 3:
        K.step3_split(rp, qi, qo, cfl, bc, bc, [1, 2, 3], O.method_array(dimensional_split=True),
                      lims, *d, dt, **kw)
    elif form == "split":
        K.step2_split(rp, qi, qo, cfl, bc, bc, [1, 2], O.method_array(dimensional_split=True),
                      lims, *d, dt, **kw)
    else:
        K.step2_unsplit(rp, qi, qo, cfl, bc, bc, [1, 2], O.method_array(transverse=2), lims, *d,
                        dt, **kw)
    torch.cuda.synchronize()
    return (q_from_device(qo) - q_from_device(co)) / scale, float(cfl.item())


@pytest.mark.parametrize("lim", [1, 3, 4])
@pytest.mark.parametrize("kind,form", [(O.ACOUSTICS, "unsplit"), (O.ACOUSTICS, "split"),
                                       (O.EULER, "unsplit"), (O.EULER, "split"),
                                       (O.SHALLOW, "unsplit"), (O.SHALLOW, "split"),
                                       (O.EULER3, "split")])
def test_large_waves_are_limited_as_small_ones(kind, form, lim):
    shape = (61, 9, 5) if kind == O.EULER3 else (67, 21)
    print("fp32 range", kind, form, lim, flush=True)
    q = _contact(kind, shape, np.random.default_rng(kind)).astype(np.float32).astype(np.float64)
    small, c_small = _step(kind, q, 1.0, lim, form)
    large, c_large = _step(kind, q, S, lim, form)
    unlimited, _ = _step(kind, q, 1.0, 0, form)
    assert np.isfinite(large).all()
    # a power of two scales every product and quotient exactly, but for a reciprocal
    # scaled on its way (1 ulp): some 50 terms of at most c max|q|, 2^-23 each
    bound = 50 * max(c_small, 0.1) * 2.0 ** -23 * np.abs(q).max()
    assert np.abs(small - unlimited).max() > 100 * bound   # the limiter matters here
    assert np.abs(large - small).max() <= bound
    assert abs(c_large - c_small) <= 2.0 ** -20 * c_small


@pytest.mark.parametrize("factor", [0.5, 1.7, 2.6])
def test_weno_weights_of_large_jumps(factor):
    """A ramp of depth whose characteristic WENO5 denominators are factor * 2^126: the
    weights of a ramp are the linear ones."""
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    mx, my, ng = 64, 9, 3
    # (13 * 0 + 3 * (2 delta)^2)^2 with delta = dh / 2, the jump of each gravity wave
    dh = 2.0 * (np.sqrt(factor) * 2.0 ** 63 / 12.0) ** 0.5
    q = np.zeros((3, mx, my), order="F")
    q[0] = (500.0 + np.arange(mx))[:, None] * dh
    q = np.asfortranarray(q.astype(np.float32).astype(np.float64))
    qbc = O.with_ghosts(q, ng)
    O.bc2(qbc, ng, [1, 1], [1, 1])
    dx, dy, dt = 1.0 / mx, 1.0 / my, 1e-8
    ref, _ = O.sharp_flux2(O.make_rp(O.SHALLOW, grav=1.0), qbc, ng, dx, dy, dt, 2)
    ref = O.interior(ref, ng)
    qi = q_to_device(q, 1)
    out = torch.empty_like(qi)
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    K.sharp2_stage(K.make_rp(O.SHALLOW, {"grav": 1.0}), 2, out, cfl, [1, 1], [1, 1], [1, 2], dt,
                   dx, dy, qi)
    torch.cuda.synchronize()
    # off the ends of the ramp, where larger denominators have no FP32 reciprocal at all
    got, ref = q_from_device(out)[:, 6:-6], ref[:, 6:-6]
    assert np.isfinite(got).all()
    # differences of fluxes g h^2 / 2, of some 20 roundings each
    flux = 0.5 * q[0].max() ** 2
    assert np.abs(got - ref).max() <= 20 * 2.0 ** -24 * flux * dt / dx


@pytest.mark.parametrize("form", ["unsplit", "split"])
@pytest.mark.parametrize("power", [120, 124, 125])
def test_stiff_acoustics(form, power):
    """Density and bulk modulus scaled by 2^power scale the impedance and the pressures, and
    leave the velocities: first-order steps (the squared norms of such waves have no FP32
    value) of an impedance of 2^(power + 1), whose double is the denominator."""
    from pyclaw_amd import kernels as K
    from pyclaw_amd.device import q_from_device, q_to_device
    mx, my, bc = 67, 21, [1, 2]
    q = np.random.default_rng(5).uniform(-0.2, 0.2, (3, mx, my)).astype(np.float32)
    d, dt = [1.0 / mx, 1.0 / my], 0.002
    outs = []
    for scale in (1.0, 2.0 ** power):
        rp = K.make_rp(O.ACOUSTICS, dict(rho=scale, bulk=4.0 * scale, cc=2.0, zz=2.0 * scale))
        qi = q_to_device(np.asfortranarray(q * np.array([scale, 1.0, 1.0])[:, None, None]), 1)
        qo, co = torch.empty_like(qi), torch.empty_like(qi)
        cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
        meth = O.method_array(order=1, dimensional_split=True) if form == "split" else \
            O.method_array(order=1, transverse=1)
        (K.step2_split if form == "split" else K.step2_unsplit)(
            rp, qi, qo, cfl, bc, bc, [1, 2], meth, [0, 0], *d, dt,
            comp_in=torch.zeros_like(qi), comp_out=co)
        torch.cuda.synchronize()
        outs.append((q_from_device(qo) - q_from_device(co)) / np.array([scale, 1.0, 1.0])[:, None, None])
    assert np.isfinite(outs[1]).all()
    # powers of two scale exactly but for a reciprocal scaled on its way (1 ulp)
    assert np.abs(outs[1] - outs[0]).max() <= 50 * 2.0 ** -23 * np.abs(q).max()
