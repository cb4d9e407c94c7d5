"""Performance cases: the time-step work a user of pyclaw_amd has it do.

A case is a dict of plain values.  Five kinds of work stand for the package's
uses, each through the solver classes:

  classic   a Controller's inner loop on ClawSolver2D's unsplit step: 16 attempts
            of the device-controlled loop (run_steps), dt from the Courant number
  split     one dimension-split step of ClawSolver2D (its default) or ClawSolver3D
  unsplit3  one unsplit step of ClawSolver3D (transverse and double-transverse
            corrections)
  sharp     SharpClawSolver2D: 16 attempts of the SSP33 loop on the periodic
            shallow-water family (characteristic WENO5, with or without the
            learned indicator), or one step of the default SSP104 integrator
            (component WENO5, acoustics)
  ensemble  16 steps of many independent unsplit Euler problems of uneven sizes

The state lives on the GPU before and after a pass, as it does between steps of a
run; a pass returns it with the time, the step size and the Courant number.

`exact` recomputes a pass in 64-bit torch from the published formulas, without
this package.
"""
import math
import os

import numpy as np
import torch

import pyclaw_amd as pyclaw
from pyclaw_amd import riemann
from pyclaw_amd.ensemble import Ensemble
from pyclaw_amd.indicator import TroubledInterfaceIndicator

STEPS = 16          # attempts of a pass: one chunk of the captured loop
GAMMA, GRAV = 1.4, 1.0
RHO, BULK = 1.0, 4.0

_CODES = {"fp64": 0, "fp64fast": 0, "fp32k": 1}     # State.device_q's type code
_BCS = {"extrap": pyclaw.BC.extrap, "periodic": pyclaw.BC.periodic, "wall": pyclaw.BC.wall}
_LIMITERS = {"minmod": pyclaw.limiters.tvd.minmod, "MC": pyclaw.limiters.tvd.MC}
_FIELDS = {"acoustics": 3, "euler": 4, "shallow": 3, "euler3": 5}
_RIEMANN = {"acoustics": riemann.acoustics_2D, "euler": riemann.euler_4wave_2D,
            "shallow": riemann.shallow_roe_with_efix_2D, "euler3": riemann.euler_3D}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # small acoustics run with solid walls: a step is a few microseconds of
        # work, so launches and each wavefront's serial chain count
        dict(name="acoustics_256_f64", kind="classic", law="acoustics", mx=256, my=256,
             precision="fp64", bc="wall", limiter="MC"),
        # the classic Euler quadrant problem, reference-equal FP64 and FP32 + Kahan
        dict(name="euler_1024_f64", kind="classic", law="euler", mx=1024, my=1024,
             precision="fp64", bc="extrap", limiter="MC"),
        dict(name="euler_1024_f32k", kind="classic", law="euler", mx=1024, my=1024,
             precision="fp32k", bc="extrap", limiter="MC"),
        # a grid larger than the caches
        dict(name="acoustics_4096_f64", kind="classic", law="acoustics", mx=4096, my=4096,
             precision="fp64", bc="wall", limiter="MC"),
        # ClawSolver2D as it comes (dimension-split), a ragged middling grid
        dict(name="shallow_split_501x487_f64", kind="split", law="shallow", mx=501, my=487,
             mz=1, precision="fp64", bc="extrap", limiter="MC"),
        # SharpClawSolver2D as it comes (SSP104, component WENO5), a small grid:
        # eleven launches and the host's step control
        dict(name="sharp104_acoustics_100_f64", kind="sharp", law="acoustics", mx=100, my=100,
             precision="fp64", bc="wall", integrator="SSP104", indicator=False),
        # the shallow-water headline grid: the reference-equal full WENO5 path ...
        dict(name="sharp_swe_2048_f64", kind="sharp", law="shallow", mx=2048, my=2048,
             precision="fp64", bc="periodic", integrator="SSP33", indicator=False),
        # ... and FP32 + Kahan with the learned indicator
        dict(name="sharp_swe_2048_f32k_ind", kind="sharp", law="shallow", mx=2048, my=2048,
             precision="fp32k", bc="periodic", integrator="SSP33", indicator=True),
        # a parameter study: many small Euler problems stepped together
        dict(name="ensemble_128_f32k", kind="ensemble", law="euler", members=128, lo=64, hi=512,
             precision="fp32k", bc="extrap", limiter="MC"),
        # 3D Euler, dimension-split: the large box in FP32 + Kahan, a ragged middling
        # one in reference-equal FP64
        dict(name="euler3d_384_f32k", kind="split", law="euler3", mx=384, my=384, mz=384,
             precision="fp32k", bc="extrap", limiter="MC"),
        dict(name="euler3d_210x170x190_f64", kind="split", law="euler3", mx=210, my=170, mz=190,
             precision="fp64", bc="extrap", limiter="MC"),
        # 3D Euler, unsplit with all transverse corrections
        dict(name="euler3d_unsplit_96x64x80_f64", kind="unsplit3", law="euler3", mx=96, my=64,
             mz=80, precision="fp64", bc="extrap", limiter="MC"),
    ]


def draw(rng):
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["classic", "classic", "split2", "split3", "unsplit3", "sharp", "sharp",
                       "sharp104", "ensemble"])
    prec = rng.choice(["fp64", "fp64", "fp64fast", "fp32k", "fp32k"])
    bc = rng.choice(["extrap", "wall", "periodic"])
    limiter = rng.choice(["MC", "MC", "minmod"])
    if kind == "classic":
        return dict(kind="classic", law=rng.choice(["acoustics", "euler", "shallow"]),
                    mx=side(64, 2800), my=side(64, 2800), precision=prec, bc=bc, limiter=limiter)
    if kind == "split2":
        return dict(kind="split", law=rng.choice(["acoustics", "euler", "shallow"]),
                    mx=side(64, 2800), my=side(64, 2800), mz=1, precision=prec, bc=bc,
                    limiter=limiter)
    if kind == "split3":
        return dict(kind="split", law="euler3", mx=side(40, 380), my=side(40, 380),
                    mz=side(40, 380), precision=prec, bc=bc, limiter=limiter)
    if kind == "unsplit3":
        return dict(kind="unsplit3", law="euler3", mx=side(24, 120), my=side(24, 120),
                    mz=side(24, 120), precision="fp64", bc=bc, limiter=limiter)
    if kind == "sharp":
        return dict(kind="sharp", law="shallow", mx=side(96, 2000), my=side(96, 2000),
                    precision=prec, bc="periodic", integrator="SSP33",
                    indicator=rng.random() < 0.5)
    if kind == "sharp104":
        return dict(kind="sharp", law=rng.choice(["acoustics", "shallow"]), mx=side(60, 600),
                    my=side(60, 600), precision=rng.choice(["fp64", "fp64fast"]), bc=bc,
                    integrator="SSP104", indicator=False)
    lo = side(32, 96)
    return dict(kind="ensemble", law="euler", members=rng.randint(24, 96), lo=lo,
                hi=rng.randint(3 * lo, 512), precision=prec, bc=bc, limiter=limiter)


def _is3d(case):
    return case["law"] == "euler3"


def _shape(case):
    """Planar array shape: (fields, [mz,] my, mx)."""
    m = _FIELDS[case["law"]]
    return (m, case["mz"], case["my"], case["mx"]) if _is3d(case) else (m, case["my"], case["mx"])


def _members(case):
    """(mx, my) of an ensemble's members, sides log-uniform; the sizes belong to
    the case, the states to the seed."""
    rng = np.random.default_rng(case["members"] + 1000 * case["lo"] + case["hi"])
    s = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), (case["members"], 2)))
    return [(int(a), int(b)) for a, b in np.rint(s)]


# Floating-point operations per cell: a classic step of a law (both directions), a
# SharpClaw operator evaluation, an unsplit 3D step.
_FLOPS = {("classic", "acoustics"): 330, ("classic", "shallow"): 900, ("classic", "euler"): 2000,
          ("ensemble", "euler"): 2000, ("split", "acoustics"): 200, ("split", "shallow"): 450,
          ("split", "euler"): 900, ("split", "euler3"): 1100, ("unsplit3", "euler3"): 5000,
          ("sharp", "acoustics"): 700, ("sharp", "shallow"): 3000}


def work(case):
    """Each step reads its state once and writes it once (the next step needs this
    one's Courant number, so a step cannot do with less); FP32 + Kahan states come
    with their compensation."""
    kind = case["kind"]
    if kind == "ensemble":
        cells = sum(a * b for a, b in _members(case))
    else:
        cells = int(np.prod(_shape(case)[1:]))
    item = 8 if precision_of(case) != "fp32k" else 2 * 4
    steps = STEPS if kind in ("classic", "ensemble") or case.get("integrator") == "SSP33" else 1
    evals = {"SSP33": 3, "SSP104": 10}.get(case.get("integrator"), 1)
    flops = _FLOPS[(kind, case["law"])]
    if case.get("indicator"):
        flops = 600          # linear reconstruction at nearly every interface
    elif case["law"] == "shallow" and case.get("integrator") == "SSP104":
        flops = 1500         # component WENO5
    return {"bytes": 2.0 * cells * _FIELDS[case["law"]] * item * steps,
            "flops": float(cells) * flops * evals * steps}


def precision_of(case):
    return case["precision"]


def tolerance(case):
    """About four times the distance from `exact` that was measured over the
    listed cases and some thirty drawn ones.  The component WENO's smoothness
    indicators are sums of products that cancel, so it is the furthest off in
    FP64; a rounding can turn a few of the indicator's flags."""
    if case["precision"] == "fp32k":
        if case.get("indicator"):
            return {"rel": 2e-6, "max": 1e-3}
        return {"rel": 8e-7, "max": 2e-4} if case["kind"] == "sharp" else {"rel": 2.5e-7,
                                                                           "max": 2e-6}
    if case.get("integrator") == "SSP104":
        return {"rel": 4e-10, "max": 4e-8}
    return {"rel": 2e-14, "max": 4e-12} if case["kind"] == "sharp" else {"rel": 4e-15,
                                                                         "max": 1e-12}


# ---------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(rng, a, b):
    return float(rng.uniform(a, b))


def _centres(n, lo=0.0, hi=1.0):
    return lo + (torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) * ((hi - lo) / n)


def _acoustics_state(mx, my, seed):
    """A pressure pulse and noise in a box, at rest."""
    rng = np.random.default_rng(seed)
    x, y = _centres(mx)[None, :], _centres(my)[:, None]
    cx, cy = rng.uniform(0.3, 0.7, 2)
    q = torch.zeros((3, my, mx), device="cuda", dtype=torch.float64)
    noise = torch.rand((my, mx), device="cuda", dtype=torch.float64, generator=_generator(seed))
    q[0] = torch.exp(-100.0 * ((x - cx) ** 2 + (y - cy) ** 2)) + 1e-3 * (2.0 * noise - 1.0)
    return q


def _quadrant_values(seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(0.5, 1.5, 4), rng.uniform(0.4, 1.0, 4), rng.uniform(-0.3, 0.3, 4),
            rng.uniform(-0.3, 0.3, 4))


def _quadrant_state(mx, my, seed):
    """Four constant gas states meeting at the centre."""
    rho, p, u, v = _quadrant_values(seed)
    x, y = _centres(mx)[None, :], _centres(my)[:, None]
    quad = ((x >= 0.5).long() + 2 * (y >= 0.5).long())
    r, pr, uu, vv = (torch.tensor(a, device="cuda", dtype=torch.float64)[quad]
                     for a in (rho, p, u, v))
    return torch.stack([r, r * uu, r * vv, pr / (GAMMA - 1.0) + 0.5 * r * (uu * uu + vv * vv)])


def _quadrant_host(mx, my, seed):
    """The same state as Solution.q takes it: (4, mx, my) on the host."""
    rho, p, u, v = _quadrant_values(seed)
    quad = ((np.arange(mx) + 0.5) / mx >= 0.5).astype(int)[:, None] \
        + 2 * ((np.arange(my) + 0.5) / my >= 0.5).astype(int)[None, :]
    r, pr, uu, vv = (a[quad] for a in (rho, p, u, v))
    q = np.empty((4, mx, my), order="F")
    q[0], q[1], q[2] = r, r * uu, r * vv
    q[3] = pr / (GAMMA - 1.0) + 0.5 * r * (uu * uu + vv * vv)
    return q


def _shallow_state(mx, my, seed):
    """Water at rest: depth 1, eight Gaussian humps, two circular dams (periodic)."""
    rng = np.random.default_rng(seed)
    x, y = _centres(mx)[None, :], _centres(my)[:, None]

    def r2(cx, cy):
        ax = torch.remainder(x - cx + 0.5, 1.0) - 0.5
        ay = torch.remainder(y - cy + 0.5, 1.0) - 0.5
        return ax * ax + ay * ay

    h = torch.ones((my, mx), device="cuda", dtype=torch.float64)
    for _ in range(8):
        amp, width = rng.uniform(0.05, 0.3), rng.uniform(0.02, 0.1)
        cx, cy = rng.uniform(0, 1, 2)
        h += amp * torch.exp(-r2(cx, cy) / (width * width))
    for _ in range(2):
        rad, jump = rng.uniform(0.05, 0.15), rng.uniform(0.1, 0.5)
        cx, cy = rng.uniform(0, 1, 2)
        h += jump * (r2(cx, cy) < rad * rad)
    q = torch.zeros((3, my, mx), device="cuda", dtype=torch.float64)
    q[0] = h
    return q


def _blast_state(mx, my, mz, seed):
    """A spherical region of higher pressure in a gas with density noise."""
    rng = np.random.default_rng(seed)
    r0, pin = _uniform(rng, 0.2, 0.4), _uniform(rng, 2.0, 4.0)
    x, y, z = _centres(mx, -1, 1), _centres(my, -1, 1), _centres(mz, -1, 1)
    r2 = x[None, None, :] ** 2 + y[None, :, None] ** 2 + z[:, None, None] ** 2
    q = torch.zeros((5, mz, my, mx), device="cuda", dtype=torch.float64)
    noise = torch.rand((mz, my, mx), device="cuda", dtype=torch.float64,
                       generator=_generator(seed))
    q[0] = 1.0 + 1e-2 * (2.0 * noise - 1.0)
    q[4] = (0.2 + (pin - 0.2) * (r2 < r0 * r0)) / (GAMMA - 1.0)
    return q


def _state(case, seed):
    law = case["law"]
    if law == "euler3":
        q = _blast_state(case["mx"], case["my"], case["mz"], seed)
    else:
        q = {"acoustics": _acoustics_state, "euler": _quadrant_state,
             "shallow": _shallow_state}[law](case["mx"], case["my"], seed)
    return q.float() if case["precision"] == "fp32k" else q


# Bounds of |u| + c of the initial states (and of the waves they raise).
_SPEED = {"acoustics": 2.0, "euler": 2.6, "shallow": 2.4, "euler3": 3.2}


def _spacing(case, mx=None, my=None):
    if _is3d(case):
        return [2.0 / case["mx"], 2.0 / case["my"], 2.0 / case["mz"]]
    return [1.0 / (mx or case["mx"]), 1.0 / (my or case["my"])]


def _cfl(case):
    """(desired, largest) Courant number."""
    if case["kind"] == "sharp":
        return (2.45, 2.5) if case["integrator"] == "SSP104" else (0.45, 0.5)
    return (0.8, 1.0)


def _first_dt(case, spacing=None):
    """A first step below the desired Courant number."""
    return 0.8 * _cfl(case)[0] * min(spacing or _spacing(case)) / _SPEED[case["law"]]


# ---------------------------------------------------------------- a user's program
def _solver(case):
    law, kind = case["law"], case["kind"]
    if kind == "sharp":
        s = pyclaw.SharpClawSolver2D(_RIEMANN[law])
        s.time_integrator = case["integrator"]
        s.char_decomp = 2 if case["integrator"] == "SSP33" else 0
        if case["indicator"]:
            s.indicator = TroubledInterfaceIndicator()
    elif _is3d(case):
        s = pyclaw.ClawSolver3D(_RIEMANN[law])
        s.dimensional_split = kind == "split"
        s.limiters = _LIMITERS[case["limiter"]]
    else:
        s = pyclaw.ClawSolver2D(_RIEMANN[law])
        s.dimensional_split = kind == "split"
        if not s.dimensional_split:
            s.transverse_waves = s.trans_cor
        s.limiters = _LIMITERS[case["limiter"]]
    s.all_bcs = _BCS[case["bc"]]
    s.precision = case["precision"]
    s.cfl_desired, s.cfl_max = _cfl(case)
    return s


def _problem_data(law):
    if law == "acoustics":
        cc = math.sqrt(BULK / RHO)
        return {"rho": RHO, "bulk": BULK, "cc": cc, "zz": RHO * cc}
    return {"grav": GRAV} if law == "shallow" else {"gamma": GAMMA}


def _solution(case, mx, my, mz=1):
    if _is3d(case):
        domain = pyclaw.Domain([-1.0] * 3, [1.0] * 3, [mx, my, mz])
    else:
        domain = pyclaw.Domain([0.0, 0.0], [1.0, 1.0], [mx, my])
    sol = pyclaw.Solution(_FIELDS[case["law"]], domain)
    sol.problem_data.update(_problem_data(case["law"]))
    return sol


def prepare(case, seed):
    solver = _solver(case)
    if case["kind"] == "ensemble":
        sols, dts = [], []
        for k, (mx, my) in enumerate(_members(case)):
            sol = _solution(case, mx, my)
            sol.q = _quadrant_host(mx, my, 1000 * int(seed) + k)
            sols.append(sol)
            dts.append(_first_dt(case, _spacing(case, mx, my)))
        return {"case": case, "ensemble": Ensemble(solver, sols, dts)}
    sol = _solution(case, case["mx"], case["my"], case.get("mz", 1))
    q = _state(case, seed)
    sol.state.set_device_q(q, torch.zeros_like(q) if case["precision"] == "fp32k" else None)
    solver.dt = solver.dt_initial = _first_dt(case)
    solver.setup(sol)
    return {"case": case, "solver": solver, "solution": sol}


def run(state):
    case = state["case"]
    if case["kind"] == "ensemble":
        ens = state["ensemble"]
        ens.run_steps(STEPS)
        # the members' two buffers: the state and the one a step before it
        return {"q": torch.cat([b[0].reshape(-1) for b in ens._bufs]),
                "q_before": torch.cat([b[1].reshape(-1) for b in ens._bufs])}
    solver, sol = state["solver"], state["solution"]
    if case["kind"] == "classic" or case.get("integrator") == "SSP33":
        solver.run_steps(sol, STEPS)
    else:
        solver.evolve_to_time(sol)
    return {"q": sol.state.device_q(_CODES[case["precision"]])[0], "t": sol.t, "dt": solver.dt,
            "cfl": solver.cfl.get_cached_max()}


# ---------------------------------------------------------------- 64-bit recomputation
# Arrays are (fields, [z,] y, x); direction n = 1, 2, 3 is axis -n, and momentum (or
# velocity) component n is field n.
class _Acoustics:
    fields, efix = 3, False
    z, c = math.sqrt(BULK * RHO), math.sqrt(BULK / RHO)

    def roe(self, ql, qr):
        return None

    def waves(self, r, d, n, lumped=False):
        a1 = (-d[0] + self.z * d[n]) / (2 * self.z)
        a2 = (d[0] + self.z * d[n]) / (2 * self.z)
        w1, w2 = torch.zeros_like(d), torch.zeros_like(d)
        w1[0], w1[n], w2[0], w2[n] = -a1 * self.z, a1, a2 * self.z, a2
        s = torch.full_like(d[0], self.c)
        return [w1, w2], [-s, s]

    def flux(self, q, n):
        f = torch.zeros_like(q)
        f[0], f[n] = BULK * q[n], q[0] / RHO
        return f


class _Shallow:
    fields, efix = 3, True

    def roe(self, ql, qr):
        sl, sr = ql[0].sqrt(), qr[0].sqrt()
        u = [None] + [(ql[k] / sl + qr[k] / sr) / (sl + sr) for k in (1, 2)]
        return u, (GRAV * 0.5 * (ql[0] + qr[0])).sqrt()

    def waves(self, r, d, n, lumped=False):
        u, a = r
        t = 3 - n
        out = []
        a1 = ((u[n] + a) * d[0] - d[n]) / (2 * a)
        a3 = (-(u[n] - a) * d[0] + d[n]) / (2 * a)
        for al, s in ((a1, u[n] - a), (None, u[n]), (a3, u[n] + a)):
            w = torch.zeros_like(d)
            if al is None:
                w[t] = d[t] - u[t] * d[0]
            else:
                w[0], w[n], w[t] = al, al * s, al * u[t]
            out.append((w, s))
        return [w for w, _ in out], [s for _, s in out]

    def speeds(self, q, n):
        return q[n] / q[0], (GRAV * q[0]).sqrt()

    def flux(self, q, n):
        un = q[n] / q[0]
        f = q * un
        f[0] = q[n]
        f[n] = f[n] + 0.5 * GRAV * q[0] ** 2
        return f


class _Euler:
    efix = True

    def __init__(self, dims):
        self.dims, self.fields = dims, dims + 2

    def pressure(self, q):
        ke = sum(q[k] ** 2 for k in range(1, self.dims + 1)) / q[0]
        return (GAMMA - 1) * (q[-1] - 0.5 * ke)

    def roe(self, ql, qr):
        sl, sr = ql[0].sqrt(), qr[0].sqrt()
        u = [None] + [(ql[k] / sl + qr[k] / sr) / (sl + sr) for k in range(1, self.dims + 1)]
        h = ((ql[-1] + self.pressure(ql)) / sl + (qr[-1] + self.pressure(qr)) / sr) / (sl + sr)
        uu = sum(v * v for v in u[1:])
        a2 = (GAMMA - 1) * (h - 0.5 * uu)
        return u, a2.sqrt(), h, uu, (GAMMA - 1) / a2

    def waves(self, r, d, n, lumped=False):
        u, a, h, uu, g1a2 = r
        ax = range(1, self.dims + 1)
        am = g1a2 * ((h - uu) * d[0] + sum(u[k] * d[k] for k in ax) - d[-1])
        al = (d[n] + (a - u[n]) * d[0] - a * am) / (2 * a)
        a1 = d[0] - am - al
        ws, ss = [], []
        for co, s, e in ((a1, u[n] - a, h - u[n] * a), (al, u[n] + a, h + u[n] * a)):
            w = torch.zeros_like(d)
            w[0], w[-1] = co, co * e
            for k in ax:
                w[k] = co * (s if k == n else u[k])
            ws.append(w)
            ss.append(s)
        ent, shear = torch.zeros_like(d), torch.zeros_like(d)
        ent[0], ent[-1] = am, am * 0.5 * uu
        for k in ax:
            ent[k] = am * u[k]
            if k != n:
                b = d[k] - u[k] * d[0]
                shear[k] = b
                shear[-1] = shear[-1] + b * u[k]
        if lumped or self.dims == 3:
            return [ws[0], ent + shear, ws[1]], [ss[0], u[n], ss[1]]
        return [ws[0], shear, ent, ws[1]], [ss[0], u[n], u[n], ss[1]]

    def speeds(self, q, n):
        return q[n] / q[0], (GAMMA * self.pressure(q) / q[0]).sqrt()


def _law(name):
    return {"acoustics": _Acoustics, "shallow": _Shallow}[name]() if name in (
        "acoustics", "shallow") else _Euler(3 if name == "euler3" else 2)


def _split(law, r, d, t):
    """The parts of d that go down and up in direction t."""
    w, s = law.waves(r, d, t, lumped=True)
    return (sum(v.clamp(max=0) * x for x, v in zip(w, s)),
            sum(v.clamp(min=0) * x for x, v in zip(w, s)))


def _solve(law, ql, qr, n):
    """Waves, speeds, left- and right-going fluctuations and the averages at the
    interfaces of ql | qr (Roe, with the Harten-Hyman entropy fix)."""
    r = law.roe(ql, qr)
    w, s = law.waves(r, qr - ql, n)
    if not law.efix:
        return w, s, sum(v.clamp(max=0) * x for x, v in zip(w, s)), \
            sum(v.clamp(min=0) * x for x, v in zip(w, s)), r
    zero = torch.zeros_like(s[0])

    def sf(a, b, mean, otherwise):
        return torch.where((a < 0) & (b > 0), mean, torch.where(otherwise < 0, otherwise, zero))

    u, c = law.speeds(ql, n)
    s0 = u - c
    u, c = law.speeds(ql + w[0], n)
    s1 = u - c
    am = sf(s0, s1, s0 * (s1 - s[0]) / (s1 - s0), s[0]) * w[0]
    u, c = law.speeds(qr - w[-1], n)
    s2 = u + c
    u, c = law.speeds(qr, n)
    s3 = u + c
    right = sf(s2, s3, s2 * (s3 - s[-1]) / (s3 - s2), s[-1]) * w[-1]
    mid = sum(v * x for x, v in zip(w[1:-1], s[1:-1]))
    am = torch.where(s[1] >= 0, am, am + mid + right)
    am = torch.where((s0 >= 0) & (s[0] > 0), torch.zeros_like(am), am)
    return w, s, am, sum(v * x for x, v in zip(w, s)) - am, r


def _pad(q, ng, bc):
    for n in range(1, q.dim()):
        m = q.shape[-n]
        i = torch.arange(-ng, m + ng, device=q.device)
        if bc == "periodic":
            j, flip = i % m, None
        elif bc == "extrap":
            j, flip = i.clamp(0, m - 1), None
        else:
            flip = (i < 0) | (i >= m)
            j = torch.where(i < 0, -1 - i, torch.where(i >= m, 2 * m - 1 - i, i))
        q = q.index_select(q.dim() - n, j)
        if flip is not None:
            sign = torch.where(flip, -1.0, 1.0).to(q.dtype)
            q[n] = q[n] * sign.reshape((-1,) + (1,) * (n - 1))
    return q


def _cut(q, n, lo, hi):
    return q.narrow(q.dim() - n, lo, q.shape[-n] - lo - hi)


class _Sweep:
    """Wave propagation along direction n of q (two ghost cells along it): the
    fluctuations and corrections at the N + 1 interfaces around N cells."""

    def __init__(self, law, q, n, dtdx, limiter):
        w, s, am, ap, r = _solve(law, _cut(q, n, 0, 1), _cut(q, n, 1, 0), n)
        self.n = n
        self.am, self.ap = _cut(am, n, 1, 1), _cut(ap, n, 1, 1)
        self.r = None if r is None else self.inner(r)
        s1 = [_cut(v, n, 1, 1) for v in s]
        self.speed = max(float(v.abs().max()) for v in s1)
        cq = 0
        for x, v in zip(w, s1):
            mid = _cut(x, n, 1, 1)
            norm = (mid * mid).sum(0)
            dot = torch.where(v > 0, (mid * _cut(x, n, 0, 2)).sum(0),
                              (mid * _cut(x, n, 2, 0)).sum(0))
            th = dot / torch.where(norm == 0, torch.ones_like(norm), norm)
            if limiter == "minmod":
                phi = th.clamp(0, 1)
            else:
                phi = torch.minimum((0.5 * (1 + th)).clamp(max=2), 2 * th).clamp(min=0)
            cq = cq + v.abs() * (1 - v.abs() * dtdx) * phi * mid
        self.cq = cq
        self.dq = -dtdx * (_cut(self.ap, n, 0, 1) + _cut(self.am, n, 1, 0)) \
            - 0.5 * dtdx * (_cut(cq, n, 1, 0) - _cut(cq, n, 0, 1))

    def inner(self, r):
        if isinstance(r, (tuple, list)):
            return [self.inner(v) for v in r]
        return r if r is None else _cut(r, self.n, 1, 1)


def _unsplit2(law, q, dt, dx, bc, limiter):
    p = _pad(q, 2, bc)
    new, cfl = q.clone(), 0.0
    for n in (1, 2):
        t = 3 - n
        dtn, dtt = dt / dx[n - 1], dt / dx[t - 1]
        s = _Sweep(law, _cut(p, t, 1, 1), n, dtn, limiter)   # slices 0 .. m+1
        cfl = max(cfl, dtn * s.speed)
        new += _cut(s.dq, t, 1, 1)
        am, ap = _split(law, s.r, s.am + s.cq, t), _split(law, s.r, s.ap - s.cq, t)
        dn, up = (-0.5 * dtn * (_cut(a, n, 1, 0) + _cut(b, n, 0, 1)) for a, b in zip(am, ap))
        g = _cut(dn, t, 1, 0) + _cut(up, t, 0, 1)            # at interfaces 1 .. m+1 of t
        new -= dtt * (_cut(g, t, 1, 0) - _cut(g, t, 0, 1))
    return new, cfl


def _split_step(law, q, dt, dx, bc, limiter):
    dims = q.dim() - 1
    p, cfl = _pad(q, 2, bc), 0.0
    for n in range(1, dims + 1):
        v = p
        if dims == 3:      # pencils 0 .. m+1 across
            for t in range(1, 4):
                if t != n:
                    v = _cut(v, t, 1, 1)
        s = _Sweep(law, v, n, dt / dx[n - 1], limiter)
        cfl = max(cfl, dt / dx[n - 1] * s.speed)
        _cut(v, n, 2, 2).add_(s.dq)
        del s
    for t in range(1, dims + 1):
        p = _cut(p, t, 2, 2)
    return p.contiguous(), cfl


def _unsplit3(law, q, dt, dx, bc, limiter):
    p = _pad(q, 2, bc)
    new, cfl = q.clone(), 0.0
    for n in (1, 2, 3):
        t1, t2 = n % 3 + 1, (n + 1) % 3 + 1
        dtn, dt1, dt2 = (dt / dx[k - 1] for k in (n, t1, t2))
        s = _Sweep(law, _cut(_cut(p, t1, 1, 1), t2, 1, 1), n, dtn, limiter)
        cfl = max(cfl, dtn * s.speed)
        cq = 0.5 * s.cq
        parts = {t: [_split(law, s.r, d, t) for d in (s.am, s.ap, cq)] for t in (t1, t2)}

        def left(x):        # a cell's left interface
            return _cut(x, n, 0, 1)

        def right(x):
            return _cut(x, n, 1, 0)

        def family(t, o, dto):
            """[down/up in t][-1, 0, 1 in o] modifications of a cell."""
            (xa, xp, xc), (za, zp, zc) = parts[t], parts[o]
            pap = _split(law, s.r, zp[1] - 3 * zc[1], t)
            pam = _split(law, s.r, za[1] + 3 * zc[1], t)
            map_ = _split(law, s.r, zp[0] - 3 * zc[0], t)
            mam = _split(law, s.r, za[0] + 3 * zc[0], t)
            k, out = dtn * dto / 6.0, []
            for i in (0, 1):
                mid = dtn * (left(xc[i]) - right(xc[i])) \
                    - 0.5 * dtn * (left(xp[i]) + right(xa[i])) \
                    + k * (left(pap[i] - map_[i]) + right(pam[i] - mam[i]))
                out.append({-1: k * (left(map_[i]) + right(mam[i])), 0: mid,
                            1: -k * (left(pap[i]) + right(pam[i]))})
            return out

        g, h = family(t1, t2, dt2), family(t2, t1, dt1)
        terms = {
            (0, 0): s.dq - dt1 * (g[1][0] - g[0][0]) - dt2 * (h[1][0] - h[0][0]),
            (-1, 0): -dt1 * g[0][0] - dt2 * (h[1][-1] - h[0][-1]),
            (-1, -1): -dt1 * g[0][-1] - dt2 * h[0][-1],
            (0, -1): -dt1 * (g[1][-1] - g[0][-1]) - dt2 * h[0][0],
            (1, -1): dt1 * g[1][-1] - dt2 * h[0][1],
            (1, 0): dt1 * g[1][0] - dt2 * (h[1][1] - h[0][1]),
            (1, 1): dt1 * g[1][1] + dt2 * h[1][1],
            (0, 1): -dt1 * (g[1][1] - g[0][1]) + dt2 * h[1][0],
            (-1, 1): -dt1 * g[0][1] + dt2 * h[1][-1]}
        for (a, b), v in terms.items():      # slice 0 .. m+1 acts on cell slice + offset
            new += _cut(_cut(v, t1, 1 - a, 1 + a), t2, 1 - b, 1 + b)
    return new, cfl


_EPS = float(np.float32(1e-36))


def _weno_component(q, n):
    """WENO5 edges (left, right) of the cells that have two neighbours on each side."""
    c = [_cut(q, n, k, 4 - k) for k in range(5)]

    def edge(a, b, m, d, e):     # the edge towards e
        w0 = 0.1 / (_EPS + 13 / 12 * (a - 2 * b + m) ** 2 + 0.25 * (a - 4 * b + 3 * m) ** 2) ** 2
        w1 = 0.6 / (_EPS + 13 / 12 * (b - 2 * m + d) ** 2 + 0.25 * (b - d) ** 2) ** 2
        w2 = 0.3 / (_EPS + 13 / 12 * (m - 2 * d + e) ** 2 + 0.25 * (3 * m - 4 * d + e) ** 2) ** 2
        return (w0 * (2 * a - 7 * b + 11 * m) + w1 * (-b + 5 * m + 2 * d)
                + w2 * (2 * m + 5 * d - e)) / (6 * (w0 + w1 + w2))

    return edge(*c[::-1]), edge(*c)


def _weno_characteristic(law, q, n):
    """Edges at the interfaces between the third and fourth of six cells: the
    right edge of the cell before, the left edge of the cell after; shallow water."""
    c = [_cut(q, n, k, 5 - k) for k in range(6)]
    u, a = law.roe(c[2], c[3])
    t = 3 - n
    d = [c[k + 1] - c[k] for k in range(5)]
    lin = (-c[1] + 7 * (c[2] + c[3]) - c[4]) / 12
    ql, qr = lin.clone(), lin.clone()

    def side(am2, am1, a0, ap1, sign):
        t1, t2, t3 = sign * (am2 - am1), sign * (am1 - a0), sign * (a0 - ap1)
        b1 = (_EPS + 13 * t1 ** 2 + 3 * (am2 - 3 * am1) ** 2) ** 2
        b2 = (_EPS + 13 * t2 ** 2 + 3 * (am1 + a0) ** 2) ** 2
        b3 = (_EPS + 13 * t3 ** 2 + 3 * (3 * a0 - ap1) ** 2) ** 2
        s1, s2, s3 = b2 * b3, 6 * b1 * b3, 3 * b1 * b2
        tot = s1 + s2 + s3
        return (s1 / tot * (t2 - t1) + (0.5 * s3 / tot - 0.25) * (t3 - t2)) / 3

    for which in range(3):
        if which == 1:
            hh = [x[t] - u[t] * x[0] for x in d]
        else:
            sg = 1 if which == 0 else -1
            hh = [sg * ((u[n] + sg * a) * x[0] - x[n]) / (2 * a) for x in d]
        ul, ur = side(hh[0], hh[1], hh[2], hh[3], 1), side(hh[4], hh[3], hh[2], hh[1], -1)
        for out, v in ((ql, ul), (qr, ur)):
            if which == 1:
                out[t] += v
            else:
                out[0] += v
                out[n] += (u[n] - a if which == 0 else u[n] + a) * v
                out[t] += u[t] * v
    return ql, qr


def _troubled(q, bc):
    """The interfaces the learned indicator gives the full WENO5, per direction:
    those one of whose components' min-max normalised stencils the network
    calls troubled (operands and hidden values in BF16), and their neighbours
    along the normal."""
    arr = np.load(os.path.join(os.path.dirname(pyclaw.__file__), "data", "indicator_swe.npy"),
                  allow_pickle=False)
    threshold, flat = float(arr[-2]), float(arr[-1])

    def part(at, *shape):
        n = int(np.prod(shape))
        w = torch.from_numpy(arr[at:at + n].astype(np.float32)).cuda()
        return w.bfloat16().double().reshape(shape)

    w1, w2, b2, w3, b3 = (part(0, 16, 32), part(512, 32, 32), part(1536, 32), part(1568, 32),
                          part(1600, 1))
    p, out = _pad(q, 3, bc), {}
    for n in (1, 2):
        v = _cut(p, 3 - n, 3, 3)
        st = torch.stack([_cut(v, n, k, 5 - k) for k in range(6)])
        lo, span = st.amin(0), st.amax(0) - st.amin(0)
        rough = span.float() > flat
        x = (st - lo) * (2.0 / torch.where(rough, span, torch.ones_like(span))) - 1.0
        x = torch.where(rough, x, torch.zeros_like(x)).bfloat16().double().reshape(6, -1)
        h = (w1[:6].T @ x + w1[6][:, None]).clamp(min=0).bfloat16().double()
        z = w3 @ (w2.T @ h + b2[:, None]).clamp(min=0) + b3
        hit = ((z.reshape(span.shape) > threshold) & rough).any(0)
        first, last = hit.narrow(2 - n, 0, 1), hit.narrow(2 - n, hit.shape[-n] - 1, 1)
        wide = torch.cat([first, hit, last], 2 - n)
        m = hit.shape[-n]
        out[n] = hit | wide.narrow(2 - n, 0, m) | wide.narrow(2 - n, 2, m)
    return out


def _operator(law, q, dt, dx, bc, characteristic, troubled=None):
    """dt L(q) and the Courant number; troubled: the interfaces of _troubled, the
    others take WENO5's linear weights."""
    out, cfl = 0, 0.0
    p = _pad(q, 3, bc)
    for n in (1, 2):
        v = _cut(p, 3 - n, 3, 3)
        if characteristic:
            before, after = _weno_characteristic(law, v, n)
            if troubled is not None:
                c = [_cut(v, n, k, 5 - k) for k in range(6)]
                lin = [(2 * a - 13 * b + 47 * m + 27 * d - 3 * e) / 60
                       for a, b, m, d, e in (c[:5], c[:0:-1])]
                before = torch.where(troubled[n], before, lin[0])
                after = torch.where(troubled[n], after, lin[1])
        else:
            lo, hi = _weno_component(v, n)                    # cells 0 .. m+1
            before, after = _cut(hi, n, 0, 1), _cut(lo, n, 1, 0)
        _, s, am, ap, _ = _solve(law, before, after, n)
        cfl = max(cfl, max(float(x.abs().max()) for x in s) * dt / dx[n - 1])
        inside = law.flux(_cut(before, n, 1, 0), n) - law.flux(_cut(after, n, 0, 1), n)
        out = out - dt / dx[n - 1] * (_cut(am, n, 1, 0) + _cut(ap, n, 0, 1) + inside)
    return out, cfl


def _exact_classic(law, q, dt, dx, case):
    """STEPS accepted attempts: (state, state before, t, dt, cfl)."""
    desired, largest = _cfl(case)
    t, old = 0.0, q
    for k in range(STEPS):
        old, (q, cfl) = q, _unsplit2(law, q, dt, dx, case["bc"], case["limiter"])
        assert cfl <= largest
        t += dt
        if k < STEPS - 1:
            dt = dt * desired / cfl
    return q, old, t, dt, cfl


def _exact_ssp33(law, q, dt, dx, case):
    desired, largest = _cfl(case)
    t = 0.0

    troubled = None

    def op(y, h):
        return _operator(law, y, h, dx, case["bc"], True, troubled)

    for k in range(STEPS):
        if case["indicator"] and k % 2 == 0:     # every second step at this Courant number
            troubled = _troubled(q, case["bc"])
        rate, cfl = op(q, dt)
        rate = rate / dt
        if k:
            dt, cfl = dt * desired / cfl, desired
        y = q + dt * rate
        d, c2 = op(y, dt)
        y = 0.75 * q + 0.25 * (y + d)
        d, c3 = op(y, dt)
        q = q / 3 + 2 / 3 * (y + d)
        cfl = max(cfl, c2, c3)
        assert cfl <= largest
        t += dt
    return q, t, dt, cfl


def _exact_ssp104(law, q, dt, dx, case):
    cfl, y, mid = 0.0, q, None
    for k in range(10):
        d, c = _operator(law, y, dt, dx, case["bc"], False)
        cfl = max(cfl, c)
        if k == 9:
            return mid + 0.6 * y + 0.1 * d, dt, dt, cfl
        y = y + d / 6
        if k == 4:
            mid = q / 25 + 0.36 * y
            y = 15 * mid - 5 * y


def exact(case, seed):
    law, dt, dx = _law(case["law"]), _first_dt(case) if case["kind"] != "ensemble" else 0, None
    if case["kind"] == "ensemble":
        now, before = [], []
        for k, (mx, my) in enumerate(_members(case)):
            q = torch.from_numpy(np.ascontiguousarray(
                _quadrant_host(mx, my, 1000 * int(seed) + k).transpose(0, 2, 1))).cuda()
            if case["precision"] == "fp32k":
                q = q.float().double()
            dx = _spacing(case, mx, my)
            r = _exact_classic(law, q, _first_dt(case, dx), dx, case)
            now.append(r[0].reshape(-1))
            before.append(r[1].reshape(-1))
        return {"q": torch.cat(now), "q_before": torch.cat(before)}
    q, dx = _state(case, seed).double(), _spacing(case)
    if case["kind"] == "classic":
        q, _, t, dt, cfl = _exact_classic(law, q, dt, dx, case)
    elif case["kind"] == "sharp":
        q, t, dt, cfl = (_exact_ssp33 if case["integrator"] == "SSP33" else _exact_ssp104)(
            law, q, dt, dx, case)
    else:
        step = _split_step if case["kind"] == "split" else _unsplit3
        t = dt
        q, cfl = step(law, q, dt, dx, case["bc"], case["limiter"])
    return {"q": q, "t": t, "dt": dt, "cfl": cfl}
