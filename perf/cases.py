"""Timed workloads of the evolution backend, each one pass through its public entry points.

Every case is a dict of plain values; its ``kind`` names the path:

* ``evolve``       BSSN method of lines: ``MoLState.steps`` on one patch (the three kernel builds);
* ``wave``         scalar wave on a Cartesian box, the same entry point;
* ``ensemble``     many small BSSN evolutions advanced together, ``Ensemble.steps``;
* ``gradient``     forward steps that record their tape, then the reverse steps of that tape;
* ``diagnostics``  the output-step driver: Ricci tensor, constraints and volume integrals.

A pass starts from the same state (``y_n`` is set to it, as a run from a checkpoint does), so a
pass repeated on a state gives the same outputs.  The state is that of a run under way: two
black holes (conformal factor and lapse of Brill-Lindquist data, masses and places from the
seed) with all 24 gridfunctions excited by smooth fields that vanish at the origin and on the
axis, ghost zones filled and det(gammabar) = det(gammahat).

``exact`` restates the discrete equations in plain torch, without the package: covariant BSSN in
spherical-like coordinates with rescaled variables, centred, upwinded and Kreiss-Oliger finite
differences, Sommerfeld or extrapolation outer boundaries, parity at the inner ones, RK4 with
det(gammabar) enforced in every stage; the reverse pass is torch's autograd through that.
"""

from __future__ import annotations

import functools
import math
import random
from fractions import Fraction

import torch

from nrpy_amd import autotune
from nrpy_amd.runtime import (
    CARTESIAN,
    OUTER_BC_EXTRAPOLATION,
    OUTER_BC_RADIATION,
    SINHSPHERICAL,
    SPHERICAL,
    SYSTEM_WAVE,
    Clock,
    Ensemble,
    MoLState,
    Patch,
    PatchConfig,
)

RECIPES = ("whole_domain", "sphere_R_gt_8")
INTEGRANDS = ("H", "MSQUARED", "LAMBDA_CONSTRAINT")


# ---------------------------------------------------------------------------- cases


def listed():
    return [
        # the head-on collision of the two_blackholes_collide example: smallest grid, all latency
        dict(name="headon_72x12x2", kind="evolve", build="spherical4", N0=72, N1=12, N2=2, outer="radiation", steps=4),
        # the same family at odd sizes, with the extrapolation outer boundary
        dict(name="spherical_151x33x10", kind="evolve", build="spherical4", N0=151, N1=33, N2=10,
             outer="extrapolation", steps=4),
        # and at the size of a resolved axisymmetric run
        dict(name="spherical_256x64x16", kind="evolve", build="spherical4", N0=256, N1=64, N2=16, outer="radiation",
             steps=4),
        # full 3D at 4th order with dissipation: the cheaper of the two 3D builds
        dict(name="sinh4_96x48x48", kind="evolve", build="sinh4", N0=96, N1=48, N2=48, outer="radiation", steps=4),
        # full 3D at 6th order: a low-resolution run, one with odd rows, and the production grid
        dict(name="sinh6_64x32x32", kind="evolve", build="sinh6", N0=64, N1=32, N2=32, outer="radiation", steps=4),
        dict(name="sinh6_127x63x62", kind="evolve", build="sinh6", N0=127, N1=63, N2=62, outer="radiation", steps=4),
        dict(name="sinh6_192x96x96", kind="evolve", build="sinh6", N0=192, N1=96, N2=96, outer="radiation", steps=4),
        # the scalar-wave example's own box, and a larger one with odd sides
        dict(name="wave_64x64x64", kind="wave", N0=64, N1=64, N2=64, steps=4),
        dict(name="wave_255x256x201", kind="wave", N0=255, N1=256, N2=201, steps=4),
        # a parameter study: 64 collisions of uneven grids advanced together
        dict(name="ensemble_64", kind="ensemble", members=64, grids=20261202, steps=4),
        # gradient of a loss through the evolution, on the grid of the lapse-extraction loss
        dict(name="gradient_96x16x4", kind="gradient", build="spherical4", N0=96, N1=16, N2=4, outer="radiation",
             steps=2),
        # an output step of a 3D run
        dict(name="diagnostics_128x64x64", kind="diagnostics", build="sinh6", N0=128, N1=64, N2=64,
             outer="radiation"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["evolve"] * 5 + ["wave", "ensemble", "gradient", "diagnostics"])
    if kind == "wave":
        return dict(kind=kind, N0=_log_int(rng, 24, 240), N1=_log_int(rng, 24, 240), N2=_log_int(rng, 24, 160), steps=4)
    if kind == "ensemble":
        return dict(kind=kind, members=_log_int(rng, 4, 64), grids=rng.randrange(1 << 30), steps=rng.choice([2, 4]))
    if kind == "gradient":
        return dict(kind=kind, build="spherical4", N0=_log_int(rng, 48, 160), N1=_log_int(rng, 8, 24),
                    N2=2 * rng.randint(1, 4), outer="radiation", steps=2)
    build = rng.choice(["spherical4", "sinh4", "sinh6"])
    outer = "radiation" if kind == "diagnostics" or rng.random() < 0.75 else "extrapolation"
    while True:
        N0, N1 = _log_int(rng, 32, 256), _log_int(rng, 8, 96)
        N2 = 2 * (_log_int(rng, 1, 12) if build == "spherical4" else _log_int(rng, 4, 48))
        if N0 * N1 * N2 <= 320_000:
            break
    case = dict(kind=kind, build=build, N0=N0, N1=N1, N2=N2, outer=outer)
    return case if kind == "diagnostics" else dict(case, steps=4)


def _members(case):
    """Grids of an ensemble: four sizes of one resolution study, drawn with the case."""
    rng = random.Random(case["grids"])
    sizes = [(48, 8, 2), (72, 12, 2), (96, 16, 4), (128, 24, 8)]
    return [dict(build="spherical4", outer="radiation", N0=n[0], N1=n[1], N2=n[2])
            for n in (rng.choice(sizes) for _ in range(case["members"]))]


class _Build:
    """Geometry and options of one of the three BSSN kernel builds."""

    def __init__(self, case):
        b = case["build"]
        self.coord = SPHERICAL if b == "spherical4" else SINHSPHERICAL
        self.size = 10.0 if b == "spherical4" else 64.0
        self.sinhw = 0.2
        self.order = 6 if b == "sinh6" else 4
        self.phi_symmetric = b == "spherical4"
        self.KO = b != "spherical4"
        self.eta, self.KO_strength, self.CFL = 2.0, 0.3, 0.5
        self.radiation = case["outer"] == "radiation"
        self.Nxx = (case["N0"], case["N1"], case["N2"])
        self.NG = self.order // 2 + 1
        self.Nx = tuple(n + 2 * self.NG for n in self.Nxx)

    def config(self):
        return PatchConfig(coord=self.coord, Nxx=self.Nxx, fd_order=self.order,
                           symmetry_axes=4 if self.phi_symmetric else 0, enable_KO=self.KO,
                           outer_bc=OUTER_BC_RADIATION if self.radiation else OUTER_BC_EXTRAPOLATION,
                           grid_physical_size=self.size, SINHW=self.sinhw, CFL_FACTOR=self.CFL, eta=self.eta,
                           KO_strength_gauge=self.KO_strength, KO_strength_nongauge=self.KO_strength,
                           setup_on_device=True)


class _State:
    def __init__(self, **kw):
        self.__dict__.update(kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "wave":
        P = Patch(PatchConfig(system=SYSTEM_WAVE, coord=CARTESIAN, Nxx=(case["N0"], case["N1"], case["N2"]),
                              fd_order=4, symmetry_axes=0, grid_physical_size=10.0, wavespeed=1.0))
        y0 = _wave_initial(case, seed, "cuda")
        return _State(case=case, y0=y0, S=MoLState(P, y0.clone()))
    if kind == "ensemble":
        members = _members(case)
        E = Ensemble([_Build(m).config() for m in members])
        autotune.apply_tuned_ensemble(E)
        y0 = [_initial(_Build(m), seed * 1009 + k, "cuda") for k, m in enumerate(members)]
        return _State(case=case, y0=y0, E=E)
    G = _Build(case)
    y0 = _initial(G, seed, "cuda")
    P = Patch(G.config())
    if kind == "gradient":
        tape = torch.empty((case["steps"], P.tape_doubles), dtype=torch.float64, device="cuda")
        return _State(case=case, y0=y0, lam0=_cotangent(G, seed, "cuda"), P=P, tape=tape, y=y0.clone(),
                      lam=torch.empty_like(y0))
    if kind == "diagnostics":
        return _State(case=case, y0=y0, P=P, aux=P.new_gfs(6), diag=P.new_gfs(6), clock=Clock(0.0, 0.0, P.dt, 0, 0))
    return _State(case=case, y0=y0, S=MoLState(P, y0.clone()))


def run(state):
    kind = state.case["kind"]
    if kind == "ensemble":
        for st, y in zip(state.E.states, state.y0):
            st.y_n.copy_(y)
        state.E.steps(state.case["steps"])
        return [st.y_n for st in state.E.states]
    if kind == "gradient":
        P, dt = state.P, state.P.dt
        state.y.copy_(state.y0)
        for tape in state.tape:
            P.MoL_step_forward_taped(state.y, dt, tape)
        state.lam.copy_(state.lam0)
        for tape in reversed(state.tape):
            P.MoL_step_adjoint_taped(tape, dt, state.lam)
        return {"y": state.y.unbind(0), "gradient": state.lam.unbind(0)}
    if kind == "diagnostics":
        integrals = state.P.diagnostics(state.clock, 1.0, state.y0, state.aux, state.diag)
        return {"fields": [state.diag[g] for g in range(6)], "integrals": integrals}
    state.S.y_n.copy_(state.y0)
    state.S.steps(state.case["steps"])
    return state.S.y_n.unbind(0)


# Operations per interior point that the point algebra and its stencils need, common
# subexpressions formed once (adds, multiplies and divides 1, a fused multiply-add 2):
# right-hand side, Ricci tensor, constraints, and the RK update with det enforcement.
_FLOPS = {"spherical4": (2956, 2274, 1429, 70), "sinh4": (4300, 2990, 1692, 70), "sinh6": (5304, 3575, 1902, 70)}


def work(case):
    """Bytes and operations of one pass.  A right-hand side needs its neighbours' stage values,
    so each of the four stages reads its 24 gridfunctions and writes the next stage's; the
    update also reads y_n (stages 2 and 3) and accumulates the running sum (written in
    stages 1 to 3, read in 2 to 4): 17 passes over the state a step, ghost zones included."""
    kind = case["kind"]
    if kind == "ensemble":
        w = [work(dict(m, kind="evolve", steps=case["steps"])) for m in _members(case)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    if kind == "wave":
        n = case["N0"] * case["N1"] * case["N2"]
        N = (case["N0"] + 4) * (case["N1"] + 4) * (case["N2"] + 4)
        return {"bytes": 17 * 2 * 8 * N * case["steps"], "flops": 4 * 40 * n * case["steps"]}
    G = _Build(case)
    n, N = math.prod(G.Nxx), math.prod(G.Nx)
    rhs, ricci, cons, rk = _FLOPS[case["build"]]
    if kind == "diagnostics":
        return {"bytes": 8 * (24 * N + 12 * n), "flops": (ricci + cons) * n}
    step = {"bytes": 17 * 24 * 8 * N, "flops": 4 * ((rhs + ricci) * n + rk * N)}
    if kind == "gradient":
        # the tape (216 values a point) is written once and read once; the reverse of the
        # algebra costs about three times the algebra
        tape = 216 * 8 * N
        return {"bytes": case["steps"] * (2 * step["bytes"] + 2 * tape), "flops": case["steps"] * 4 * step["flops"]}
    return {k: v * case["steps"] for k, v in step.items()}


def tolerance(case):
    """About four times the largest difference from ``exact`` over these ranges.  The rounding of
    a second derivative grows with 1 / dx^2 / r^2, so the small fields (aDD00, aDD22 of the
    SinhSpherical grids, the Hamiltonian constraint) carry more of it than the others."""
    if case["kind"] == "wave":
        return {"rel": 4e-12, "max": 1e-9}
    if case["kind"] == "ensemble":  # a member's 24 gridfunctions are one output
        return {"rel": 1e-14, "max": 1e-12}
    if case["kind"] == "diagnostics":
        return {"rel": 1e-6, "max": 1.5e-4}
    if case["build"] == "spherical4":
        return {"rel": 1e-11, "max": 3e-10}
    return {"rel": 1.2e-9, "max": 2e-7}


# ---------------------------------------------------------------------------- initial states

EVOL = ["aDD00", "aDD01", "aDD02", "aDD11", "aDD12", "aDD22", "alpha", "betU0", "betU1", "betU2", "cf",
        "hDD00", "hDD01", "hDD02", "hDD11", "hDD12", "hDD22", "lambdaU0", "lambdaU1", "lambdaU2", "trK",
        "vetU0", "vetU1", "vetU2"]
A, ALPHA, B, CF, H, LAM, TRK, V = 0, 6, 7, 10, 11, 17, 20, 21
SYM = {(0, 0): 0, (0, 1): 1, (0, 2): 2, (1, 1): 3, (1, 2): 4, (2, 2): 5}
F64 = torch.float64


def _grid(G, device):
    """Coordinates of all points (three 1D tensors) and the reference metric's scale factors."""
    lo, hi = (0.0, 0.0, -math.pi), (G.size if G.coord == SPHERICAL else 1.0, math.pi, math.pi)
    dxx = [(hi[d] - lo[d]) / G.Nxx[d] for d in range(3)]
    xx = [lo[d] + (torch.arange(G.Nx[d], dtype=F64, device=device) - G.NG + 0.5) * dxx[d] for d in range(3)]
    return xx, dxx


def _radius(G, x):
    """r(xx0) and its first three derivatives."""
    if G.coord == SPHERICAL:
        return x, torch.ones_like(x), torch.zeros_like(x), torch.zeros_like(x)
    w = G.sinhw
    c = G.size / math.sinh(1 / w)
    s, ch = torch.sinh(x / w), torch.cosh(x / w)
    return c * s, c / w * ch, c / w**2 * s, c / w**3 * ch


@functools.lru_cache(maxsize=4)
def _inner_map(Nxx, NG, device):
    """Source index of every point under the parity conditions (itself for interior and pure
    outer points) and the sign of each of the ten parity types there."""
    Nx = [n + 2 * NG for n in Nxx]
    i2, i1, i0 = torch.meshgrid(*[torch.arange(n) for n in reversed(Nx)], indexing="ij")
    th0, ph0 = (i1 - NG + 0.5) * (math.pi / Nxx[1]), (i2 - NG + 0.5) * (2 * math.pi / Nxx[2])
    j0, j1, j2 = i0.clone(), i1.clone(), i2.clone()
    through = j0 < NG  # r < 0: the antipodal direction
    j0 = torch.where(through, 2 * NG - 1 - j0, j0)
    j1 = torch.where(through, 2 * NG + Nxx[1] - 1 - j1, j1)
    j2 = torch.where(through, j2 + Nxx[2] // 2, j2)
    for _ in range(1 + (2 * NG) // Nxx[1]):  # across the axis (more than once on very coarse grids)
        over = (j1 < NG) | (j1 >= NG + Nxx[1])
        j1 = torch.where(j1 < NG, 2 * NG - 1 - j1, torch.where(j1 >= NG + Nxx[1], 2 * (NG + Nxx[1]) - 1 - j1, j1))
        j2 = torch.where(over, j2 + Nxx[2] // 2, j2)
    j2 = NG + torch.remainder(j2 - NG, Nxx[2])
    th1, ph1 = (j1 - NG + 0.5) * (math.pi / Nxx[1]), (j2 - NG + 0.5) * (2 * math.pi / Nxx[2])
    c = torch.cos(ph0 - ph1)
    dots = [torch.sin(th0) * torch.sin(th1) * c + torch.cos(th0) * torch.cos(th1),
            torch.cos(th0) * torch.cos(th1) * c + torch.sin(th0) * torch.sin(th1), c]
    s = [torch.sign(d).to(F64) for d in dots]
    one = torch.ones_like(s[0])
    types = [one] + s + [s[0] * s[0], s[0] * s[1], s[0] * s[2], s[1] * s[1], s[1] * s[2], s[2] * s[2]]
    src = j0 + Nx[0] * (j1 + Nx[1] * j2)
    per_gf = torch.stack([types[_parity(g)] for g in EVOL])
    return src.reshape(-1).to(device), per_gf.reshape(24, -1).to(device)


def _parity(gf):
    if gf[-1].isdigit() and gf[-2].isdigit():
        return 4 + SYM[(int(gf[-2]), int(gf[-1]))]
    return int(gf[-1]) + 1 if gf[-1].isdigit() else 0


def _apply_inner(G, f):
    src, sign = _inner_map(G.Nxx, G.NG, str(f.device))
    return (sign * f.reshape(24, -1)[:, src]).reshape(f.shape)


def _initial(G, seed, device):
    rng = random.Random(seed)
    xx, _ = _grid(G, device)
    r = _radius(G, xx[0])[0].abs()[None, None, :]
    th, ph = xx[1][None, :, None], xx[2][:, None, None]
    st = torch.sin(th)
    X, Y, Z = r * st * torch.cos(ph), r * st * torch.sin(ph), r * torch.cos(th)
    psi = 1.0
    for side in (1, -1):
        m, z = rng.uniform(0.3, 0.7), side * rng.uniform(0.3, 1.0)
        x = 0.0 if G.phi_symmetric else side * rng.uniform(-0.3, 0.3)
        psi = psi + m / (2 * torch.sqrt((X - x) ** 2 + Y**2 + (Z - z) ** 2))
    w = 1 / psi**2
    reach = r * r / (1 + r * r) * torch.exp(-((r / 20) ** 2)) * st * st
    y = []
    for g in EVOL:
        a, k, p, q = rng.uniform(-1, 1), rng.uniform(0.3, 1.0), rng.uniform(0, 6), rng.uniform(0, 6)
        m = 0 if G.phi_symmetric else rng.randint(0, 2)
        mode = 1e-2 * a * reach * torch.sin(k * r + p) * torch.cos(m * ph + q)
        y.append(w * (1 + mode) if g in ("alpha", "cf") else mode.expand(*reversed(G.Nx)))
    y = torch.stack([t.expand(*reversed(G.Nx)) for t in y])
    return _enforce_det(G, _apply_inner(G, y)).contiguous()


def _cotangent(G, seed, device):
    """Adjoint of the state after the last step: a smooth weight on every gridfunction inside."""
    rng = random.Random(seed + 77)
    xx, _ = _grid(G, device)
    NG = G.NG
    lam = torch.zeros((24, *reversed(G.Nx)), dtype=F64, device=device)
    r, th = xx[0][None, None, :], xx[1][None, :, None]
    for g in range(24):
        f = rng.uniform(-1, 1) * torch.sin(th) * torch.sin(rng.uniform(0.3, 1.0) * r + rng.uniform(0, 6))
        f = f.expand(*reversed(G.Nx))
        lam[g, NG:-NG, NG:-NG, NG:-NG] = f[NG:-NG, NG:-NG, NG:-NG]
    return lam


def _wave_initial(case, seed, device):
    """A few Gaussian pulses inside the box, moving and at rest, on all points."""
    rng = random.Random(seed)
    N = (case["N0"], case["N1"], case["N2"])
    xx = [-10.0 + (torch.arange(n + 4, dtype=F64, device=device) - 2 + 0.5) * (20.0 / n) for n in N]
    x, y, z = xx[0][None, None, :], xx[1][None, :, None], xx[2][:, None, None]
    u = v = 0.0
    for _ in range(3):
        c = [rng.uniform(-4, 4) for _ in range(3)]
        bump = torch.exp(-((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2) / (2 * rng.uniform(0.8, 1.6) ** 2))
        u, v = u + rng.uniform(0.5, 1.0) * bump, v + rng.uniform(-1.0, 1.0) * bump
    return torch.stack([2.0 + u, v]).contiguous()


# ---------------------------------------------------------------------------- the equations


def _weights(offsets, deriv):
    """Finite-difference weights of the ``deriv``-th derivative on integer offsets."""
    n = len(offsets)
    M = [[Fraction(o) ** i for o in offsets] + [Fraction(math.factorial(deriv) if i == deriv else 0)] for i in range(n)]
    for i in range(n):
        p = next(r for r in range(i, n) if M[r][i])
        M[i], M[p] = M[p], M[i]
        M[i] = [v / M[i][i] for v in M[i]]
        for r in range(n):
            if r != i and M[r][i]:
                M[r] = [a - M[r][i] * b for a, b in zip(M[r], M[i])]
    return [(o, M[i][n]) for i, o in enumerate(offsets) if M[i][n]]


@functools.lru_cache(maxsize=None)
def _stencils(order):
    h = order // 2
    ko = [(o, w * Fraction(-1) ** ((order + 4) // 2) / 2 ** (order + 2))
          for o, w in _weights(range(-h - 1, h + 2), order + 2)]
    return {"d": _weights(range(-h, h + 1), 1), "dd": _weights(range(-h, h + 1), 2),
            "up": _weights(range(-h + 1, h + 2), 1), "dn": _weights(range(-h - 1, h), 1), "ko": ko}


def _is0(x):
    return isinstance(x, (int, float)) and x == 0


def _mul(*a):
    if any(_is0(x) for x in a):
        return 0
    return functools.reduce(lambda p, q: p * q, a)


def _sum(terms):
    t = [x for x in terms if not _is0(x)]
    return functools.reduce(lambda p, q: p + q, t) if t else 0


R3 = range(3)


class _Metric:
    """Reference metric of the interior points: scale factors s_i, ReDD = s_i s_j, Christoffels."""

    def __init__(self, G, device, interior):
        xx, self.dxx = _grid(G, device)
        if interior:
            xx = [x[G.NG:-G.NG] for x in xx]
        f0, f0p, f0pp, f0ppp = (t[None, None, :] for t in _radius(G, xx[0]))
        f1, f1p, f1pp = torch.sin(xx[1])[None, :, None], torch.cos(xx[1])[None, :, None], -torch.sin(xx[1])[None, :, None]
        flat = G.coord == SPHERICAL
        z2, z3 = (0, 0) if flat else (f0pp, f0ppp)
        self.s = s = [f0p, f0, f0 * f1]
        self.sd = sd = [[z2, 0, 0], [f0p, 0, 0], [f0p * f1, f0 * f1p, 0]]
        sdd = [[[0] * 3 for _ in R3] for _ in R3]
        sdd[0][0][0], sdd[1][0][0] = z3, z2
        sdd[2][0][0], sdd[2][0][1], sdd[2][1][0], sdd[2][1][1] = _mul(z2, f1), f0p * f1p, f0p * f1p, f0 * f1pp
        self.sdd = sdd
        self.Re = [[s[i] * s[j] for j in R3] for i in R3]
        self.Red = [[[_sum([_mul(sd[i][k], s[j]), _mul(s[i], sd[j][k])]) for k in R3] for j in R3] for i in R3]
        self.Redd = [[[[_sum([_mul(sdd[i][k][l], s[j]), _mul(sd[i][k], sd[j][l]), _mul(sd[i][l], sd[j][k]),
                              _mul(s[i], sdd[j][k][l])]) for l in R3] for k in R3] for j in R3] for i in R3]
        self.ReU = [1 / s[i] for i in R3]
        self.ReUd = [[_mul(-1, sd[i][k], self.ReU[i], self.ReU[i]) for k in R3] for i in R3]
        self.ReUdd = [[[_sum([_mul(2, sd[i][k], sd[i][l], self.ReU[i] ** 3),
                              _mul(-1, sdd[i][k][l], self.ReU[i] ** 2)]) for l in R3] for k in R3] for i in R3]

        def g(i, j, k):
            return self.Red[i][i][k] if i == j else 0

        def gg(i, j, k, l):
            return self.Redd[i][i][k][l] if i == j else 0

        inv = [0.5 / self.Re[i][i] for i in R3]
        self.Gam = [[[_mul(inv[i], _sum([g(i, j, k), g(i, k, j), _mul(-1, g(j, k, i))])) for k in R3] for j in R3]
                    for i in R3]
        self.Gamd = [[[[_sum([_mul(-1, g(i, i, l), 1 / self.Re[i][i], self.Gam[i][j][k]),
                              _mul(inv[i], _sum([gg(i, j, k, l), gg(i, k, j, l), _mul(-1, gg(j, k, i, l))]))])
                        for l in R3] for k in R3] for j in R3] for i in R3]
        # first and second derivatives of log det(ghat)
        self.L = [_sum([_mul(2, sd[i][k], self.ReU[i]) for i in R3]) for k in R3]
        self.Ld = [[_sum([_mul(2, sdd[i][k][l], self.ReU[i]) for i in R3]
                         + [_mul(-2, sd[i][k], sd[i][l], self.ReU[i] ** 2) for i in R3]) for l in R3] for k in R3]


class _Point:
    """Derivatives and conformal tensors of a state at the interior points."""

    def __init__(self, G, M, y):
        self.G, self.M, self.y = G, M, y
        self.st = _stencils(G.order)
        self.inv = [1 / d for d in M.dxx]
        h = [[y_c(self, H + SYM[min(i, j), max(i, j)]) for j in R3] for i in R3]
        self.h = h
        self.hd = [[[self.d(self.sym(H, i, j), k) for k in R3] for j in R3] for i in R3]
        self.gDD = [[_sum([h[i][j] * M.Re[i][j], M.Re[i][i] if i == j else 0]) for j in R3] for i in R3]
        g = self.gDD
        det = (g[0][0] * (g[1][1] * g[2][2] - g[1][2] ** 2) - g[0][1] * (g[0][1] * g[2][2] - g[1][2] * g[0][2])
               + g[0][2] * (g[0][1] * g[1][2] - g[1][1] * g[0][2]))
        u = [[None] * 3 for _ in R3]
        for i in R3:
            for j in R3:
                a, b, c, d = (i + 1) % 3, (i + 2) % 3, (j + 1) % 3, (j + 2) % 3
                u[j][i] = (g[a][c] * g[b][d] - g[a][d] * g[b][c]) / det
        self.gUU = u
        self.gd = [[[_sum([M.Red[i][i][k] if i == j else 0, _mul(h[i][j], M.Red[i][j][k]),
                           _mul(self.hd[i][j][k], M.Re[i][j])]) for k in R3] for j in R3] for i in R3]
        low = [[[_mul(0.5, _sum([self.gd[m][k][l], self.gd[m][l][k], _mul(-1, self.gd[k][l][m])])) for l in R3]
                for k in R3] for m in R3]
        self.Gam = [[[_sum([_mul(u[i][m], low[m][k][l]) for m in R3]) for l in R3] for k in R3] for i in R3]
        self.DG = [[[_sum([self.Gam[i][j][k], _mul(-1, M.Gam[i][j][k])]) for k in R3] for j in R3] for i in R3]
        self.DGU = [_sum([_mul(u[j][k], self.DG[i][j][k]) for j in R3 for k in R3]) for i in R3]
        self.a = [[y_c(self, self.sym(A, i, j)) for j in R3] for i in R3]
        self.ADD = [[self.a[i][j] * M.Re[i][j] for j in R3] for i in R3]
        self.AUD = [[_sum([u[i][k] * self.ADD[k][j] for k in R3]) for j in R3] for i in R3]
        self.AUU = [[_sum([self.AUD[i][l] * u[l][j] for l in R3]) for j in R3] for i in R3]
        self.alpha, self.cf, self.trK = y_c(self, ALPHA), y_c(self, CF), y_c(self, TRK)
        cfd = [self.d(CF, k) for k in R3]
        self.phid = [_mul(-0.5, cfd[k], 1 / self.cf) for k in R3]
        phidd = [[_mul(0.5, _sum([_mul(-1, self.dd(CF, i, j)), _mul(cfd[i], cfd[j], 1 / self.cf)]), 1 / self.cf)
                  for j in R3] for i in R3]
        self.phiBB = [[_sum([phidd[i][j]] + [_mul(-1, self.Gam[k][i][j], self.phid[k]) for k in R3]) for j in R3]
                      for i in R3]

    @staticmethod
    def sym(base, i, j):
        return base + SYM[min(i, j), max(i, j)]

    def shift(self, f, off):
        NG, Nx = self.G.NG, self.G.Nx
        return f[NG + off[2]:Nx[2] - NG + off[2], NG + off[1]:Nx[1] - NG + off[1], NG + off[0]:Nx[0] - NG + off[0]]

    def line(self, gf, op, k):
        off = [0, 0, 0]
        acc = 0
        for o, w in self.st[op]:
            off[k] = o
            acc = acc + float(w) * self.shift(self.y[gf], off)
        return acc * self.inv[k]

    def none(self, k):
        return k == 2 and self.G.phi_symmetric

    def d(self, gf, k):
        return 0 if self.none(k) else self.line(gf, "d", k)

    def dd(self, gf, k, l):
        if self.none(k) or self.none(l):
            return 0
        if k == l:
            return self.line(gf, "dd", k) * self.inv[k]
        k, l = min(k, l), max(k, l)
        acc = 0
        for o, w in self.st["d"]:
            for q, v in self.st["d"]:
                off = [0, 0, 0]
                off[k], off[l] = o, q
                acc = acc + float(w * v) * self.shift(self.y[gf], off)
        return acc * (self.inv[k] * self.inv[l])

    def up(self, gf, k):
        if self.none(k):
            return 0
        return torch.where(self.beta[k] > 0, self.line(gf, "up", k), self.line(gf, "dn", k))

    def ko(self, gf, k):
        return self.line(gf, "ko", k) if self.G.KO and not self.none(k) else 0

    def ricci(self):
        M, h, hd, u, DG, g = self.M, self.h, self.hd, self.gUU, self.DG, self.gDD
        eps = [[h[i][j] * M.Re[i][j] for j in R3] for i in R3]
        epsd = [[[_sum([_mul(hd[i][j][k], M.Re[i][j]), _mul(h[i][j], M.Red[i][j][k])]) for k in R3] for j in R3]
                for i in R3]
        second = {}
        for i, j in SYM:
            for k, l in SYM:
                second[i, j, k, l] = self.dd(self.sym(H, i, j), k, l)
        epsdd = [[[[_sum([_mul(second[min(i, j), max(i, j), min(k, l), max(k, l)], M.Re[i][j]),
                          _mul(hd[i][j][k], M.Red[i][j][l]), _mul(hd[i][j][l], M.Red[i][j][k]),
                          _mul(h[i][j], M.Redd[i][j][k][l])]) for l in R3] for k in R3] for j in R3] for i in R3]
        Gh, Ghd = M.Gam, M.Gamd
        D = [[[_sum([epsd[i][j][l]] + [_mul(-1, Gh[m][i][l], eps[m][j]) for m in R3]
                    + [_mul(-1, Gh[m][j][l], eps[i][m]) for m in R3]) for l in R3] for j in R3] for i in R3]
        lamd = [[_sum([_mul(self.d(LAM + k, j), M.ReU[k]), _mul(y_c(self, LAM + k), M.ReUd[k][j])]
                      + [_mul(Gh[k][m][j], y_c(self, LAM + m), M.ReU[m]) for m in R3]) for j in R3] for k in R3]
        DGD = [[[_sum([_mul(g[i][m], DG[m][j][k]) for m in R3]) for k in R3] for j in R3] for i in R3]
        out = {}
        for i, j in SYM:
            t = []
            for l in R3:
                for k in R3:
                    d1 = [epsdd[i][j][l][k]]
                    for m in R3:
                        d1 += [_mul(-1, Ghd[m][i][l][k], eps[m][j]), _mul(-1, Gh[m][i][l], epsd[m][j][k]),
                               _mul(-1, Ghd[m][j][l][k], eps[i][m]), _mul(-1, Gh[m][j][l], epsd[i][m][k]),
                               _mul(-1, Gh[m][l][k], D[i][j][m]), _mul(-1, Gh[m][i][k], D[m][j][l]),
                               _mul(-1, Gh[m][j][k], D[i][m][l])]
                    t.append(_mul(-0.5, u[k][l], _sum(d1)))
                    for m in R3:
                        t.append(_mul(u[k][l], _sum([_mul(DG[m][k][i], DGD[j][m][l]), _mul(DG[m][k][j], DGD[i][m][l]),
                                                     _mul(DG[m][i][k], DGD[m][j][l])])))
            for k in R3:
                t += [_mul(0.5, g[k][i], lamd[k][j]), _mul(0.5, g[k][j], lamd[k][i]),
                      _mul(0.5, self.DGU[k], _sum([DGD[i][j][k], DGD[j][i][k]]))]
            out[i, j] = _sum(t)
        self.R = [[out[min(i, j), max(i, j)] for j in R3] for i in R3]
        return self.R

    def rhs(self):
        M, u, g, Gm, DG = self.M, self.gUU, self.gDD, self.Gam, self.DG
        alpha, cf, trK, ADD, AUD, AUU, phid = self.alpha, self.cf, self.trK, self.ADD, self.AUD, self.AUU, self.phid
        vet, bet, lam = ([y_c(self, b + i) for i in R3] for b in (V, B, LAM))
        self.beta = beta = [vet[i] * M.ReU[i] for i in R3]
        BU, LU = [bet[i] * M.ReU[i] for i in R3], [lam[i] * M.ReU[i] for i in R3]
        vd = [[self.d(V + i, j) for j in R3] for i in R3]
        bd = [[_sum([_mul(vd[i][j], M.ReU[i]), _mul(vet[i], M.ReUd[i][j])]) for j in R3] for i in R3]
        bdd = [[[_sum([_mul(self.dd(V + i, j, k), M.ReU[i]), _mul(vd[i][j], M.ReUd[i][k]), _mul(vd[i][k], M.ReUd[i][j]),
                       _mul(vet[i], M.ReUdd[i][j][k])]) for k in R3] for j in R3] for i in R3]

        def upU(base, f):
            return [[_sum([_mul(self.up(base + i, j), M.ReU[i]), _mul(f[i], M.ReUd[i][j])]) for j in R3] for i in R3]

        div = _sum([bd[k][k] for k in R3] + [_mul(0.5, beta[k], M.L[k]) for k in R3])
        trA = _sum([u[i][j] * ADD[i][j] for i in R3 for j in R3])
        ad = [self.d(ALPHA, k) for k in R3]
        aBB = [[_sum([self.dd(ALPHA, i, j)] + [_mul(-1, Gm[k][i][j], ad[k]) for k in R3]) for j in R3] for i in R3]
        out = [None] * 24

        def advect(base, f, i, j, unit):
            """beta^k partial_k (upwinded) plus the two terms of the Lie derivative of a tensor."""
            t = []
            for k in R3:
                part = [_mul(self.up(self.sym(base, i, j), k), M.Re[i][j]), _mul(y_c(self, self.sym(base, i, j)), M.Red[i][j][k])]
                if unit and i == j:
                    part.append(M.Red[i][i][k])
                t += [_mul(beta[k], _sum(part)), _mul(bd[k][i], f[k][j]), _mul(bd[k][j], f[i][k])]
            return t

        X = [[_sum([_mul(-2, alpha, self.phiBB[i][j]), _mul(4, alpha, phid[i], phid[j]), _mul(2, ad[i], phid[j]),
                    _mul(2, ad[j], phid[i]), _mul(-1, aBB[i][j]), _mul(alpha, self.R[i][j])]) for j in R3] for i in R3]
        X = [[X[min(i, j)][max(i, j)] for j in R3] for i in R3]
        trX = _sum([_mul(u[i][j], X[i][j]) for i in R3 for j in R3])
        for i, j in SYM:
            gr = _sum(advect(H, g, i, j, True) + [2 / 3 * g[i][j] * (alpha * trA - div), -2 * alpha * ADD[i][j]])
            ar = _sum(advect(A, ADD, i, j, False) + [-2 / 3 * ADD[i][j] * div, alpha * ADD[i][j] * trK]
                      + [-2 * alpha * ADD[i][k] * AUD[k][j] for k in R3]
                      + [cf * cf * _sum([X[i][j], -1 / 3 * g[i][j] * trX])])
            out[self.sym(H, i, j)], out[self.sym(A, i, j)] = gr / M.Re[i][j], ar / M.Re[i][j]
        out[CF] = _sum([-1 / 3 * cf * (div - alpha * trK)] + [_mul(beta[k], self.up(CF, k)) for k in R3])
        out[TRK] = _sum([alpha * trK * trK / 3] + [_mul(beta[k], self.up(TRK, k)) for k in R3]
                        + [_mul(-1, cf * cf, u[i][j], _sum([aBB[i][j], _mul(2, ad[j], phid[i])])) for i in R3 for j in R3]
                        + [alpha * ADD[i][j] * AUU[i][j] for i in R3 for j in R3])
        out[ALPHA] = _sum([-2 * alpha * trK] + [_mul(beta[k], self.up(ALPHA, k)) for k in R3])
        Lup, Bup, bup = upU(LAM, lam), upU(B, bet), upU(V, vet)
        Gh, Ghd = M.Gam, M.Gamd
        ddiv = [_sum([bdd[k][k][m] for k in R3] + [_mul(0.5, bd[k][m], M.L[k]) for k in R3]
                     + [_mul(0.5, beta[k], M.Ld[k][m]) for k in R3]) for m in R3]
        trKd = [self.d(TRK, k) for k in R3]
        for i in R3:
            t = [_mul(beta[k], Lup[i][k]) for k in R3] + [_mul(-1, bd[i][k], LU[k]) for k in R3]
            for j in R3:
                for k in R3:
                    q = [bdd[i][k][j]]
                    for m in R3:
                        q += [_mul(Ghd[i][m][k][j], beta[m]), _mul(Gh[i][m][k], bd[m][j]), _mul(Gh[i][m][j], bd[m][k]),
                              _mul(-1, Gh[m][k][j], bd[i][m])]
                        for d in R3:
                            q += [_mul(Gh[i][d][j], Gh[d][m][k], beta[m]), _mul(-1, Gh[d][k][j], Gh[i][m][d], beta[m])]
                    t += [_mul(u[j][k], _sum(q)), _mul(2, alpha, AUU[j][k], DG[i][j][k])]
            t += [_mul(2 / 3, self.DGU[i], div)]
            for m in R3:
                t += [_mul(1 / 3, u[i][m], ddiv[m]), _mul(-2, AUU[i][m], _sum([ad[m], _mul(-6, alpha, phid[m])])),
                      _mul(-4 / 3, alpha, u[i][m], trKd[m])]
            lr = _sum(t)
            vr = [BU[i]] + [_mul(beta[j], bup[i][j]) for j in R3]
            br = [0.75 * lr, -self.G.eta * BU[i]]
            for j in R3:
                br += [_mul(beta[j], Bup[i][j]), _mul(-0.75, beta[j], Lup[i][j])]
                for m in R3:
                    vr.append(_mul(beta[j], Gm[i][m][j], beta[m]))
                    br += [_mul(beta[j], Gm[i][m][j], BU[m]), _mul(-0.75, beta[j], Gm[i][m][j], LU[m])]
            out[LAM + i], out[V + i], out[B + i] = lr * M.s[i], _sum(vr) * M.s[i], _sum(br) * M.s[i]
        if self.G.KO:
            out = [_sum([f] + [_mul(self.G.KO_strength, self.ko(n, k), M.ReU[k]) for k in R3]) for n, f in enumerate(out)]
        shape = tuple(reversed(self.G.Nxx))
        return torch.nn.functional.pad(torch.stack([f.expand(shape) for f in out]), (self.G.NG,) * 6)

    def constraints(self):
        u, Gm, AUU = self.gUU, self.Gam, self.AUU
        Ham = _sum([2 / 3 * self.trK**2] + [-self.ADD[i][j] * AUU[i][j] for i in R3 for j in R3]
                   + [_mul(self.cf**2, u[i][j], _sum([self.R[i][j], _mul(-8, self.phid[i], self.phid[j]),
                                                      _mul(-8, self.phiBB[i][j])])) for i in R3 for j in R3])
        M = self.M
        Ad = [[[_sum([_mul(M.Red[i][j][k], self.a[i][j]), _mul(M.Re[i][j], self.d(self.sym(A, i, j), k))]
                     + [_mul(-1, Gm[l][k][i], self.ADD[l][j]) for l in R3]
                     + [_mul(-1, Gm[l][k][j], self.ADD[i][l]) for l in R3]) for k in R3] for j in R3] for i in R3]
        kd = [self.d(TRK, k) for k in R3]
        MU = []
        for i in R3:
            t = []
            for j in R3:
                t += [_mul(6, AUU[i][j], self.phid[j]), _mul(-2 / 3, u[i][j], kd[j])]
                for k in R3:
                    t += [_mul(u[i][k], u[j][l], Ad[k][l][j]) for l in R3]
            MU.append(self.cf**2 * _sum(t))
        M2 = _sum([self.gDD[i][j] * MU[i] * MU[j] for i in R3 for j in R3]) / self.cf**2
        L = [_sum([y_c(self, LAM + i) * M.ReU[i], _mul(-1, self.DGU[i])]) for i in R3]
        lam = torch.sqrt(_sum([self.gDD[i][j] * L[i] * L[j] for i in R3 for j in R3]))
        return [Ham, *MU, M2, lam]


def y_c(p, gf):
    return p.shift(p.y[gf], (0, 0, 0))


def _enforce_det(G, y):
    M = _Metric(G, y.device, interior=False)
    h = [[y[H + SYM[min(i, j), max(i, j)]] + (1.0 if i == j else 0.0) for j in R3] for i in R3]
    det = (h[0][0] * (h[1][1] * h[2][2] - h[1][2] ** 2) - h[0][1] * (h[0][1] * h[2][2] - h[1][2] * h[0][2])
           + h[0][2] * (h[0][1] * h[1][2] - h[1][1] * h[0][2]))
    fac = torch.pow(torch.abs(det), -1 / 3)
    new = [fac * h[i][j] - (1.0 if i == j else 0.0) for i, j in SYM]
    return torch.cat([y[:H], torch.stack(new), y[H + 6:]])


def _radiation(G, f, k):
    """Sommerfeld condition on the outer layers of the right-hand side, innermost layer first."""
    xx, dxx = _grid(G, f.device)
    r, drdx = _radius(G, xx[0])[:2]
    c = torch.ones(24, dtype=F64, device=f.device)
    inf = torch.zeros(24, dtype=F64, device=f.device)
    c[ALPHA], inf[ALPHA], inf[CF] = math.sqrt(2.0), 1.0, 1.0
    c, inf = c[:, None, None], inf[:, None, None]
    NG, N0 = G.NG, G.Nx[0]
    f = f[:, NG:-NG, NG:-NG]

    def dr(i):
        shift = N0 - 3 - i if i > N0 - 3 else -1
        acc = 0
        for o, w in _weights(range(shift - 2, shift + 3), 1):
            acc = acc + float(w) * f[..., i + o]
        return acc / dxx[0] / drdx[i]

    cols = [k[:, NG:-NG, NG:-NG, N0 - NG - 1]]
    for i in range(N0 - NG, N0):
        j = i - 1
        tail = r[j] ** 3 * (cols[-1] + c * (dr(j) + (f[..., j] - inf) / r[j]))
        cols.append(-c * (dr(i) + (f[..., i] - inf) / r[i]) + tail / r[i] ** 3)
    outer = torch.nn.functional.pad(torch.stack(cols[1:], -1), (0, 0, NG, NG, NG, NG))
    return torch.cat([k[..., :N0 - NG], outer], -1)


def _extrapolate(f, n, dim):
    """n layers past the end of dim, each the quadratic through the three before it."""
    cols = list(torch.unbind(f.narrow(dim, f.shape[dim] - 3, 3), dim))
    for _ in range(n):
        cols.append(3 * cols[-1] - 3 * cols[-2] + cols[-3])
    return torch.cat([f, torch.stack(cols[3:], dim)], dim)


def _step(G, y, dt):
    M = _Metric(G, y.device, interior=True)

    def slope(stage):
        p = _Point(G, M, stage)
        p.ricci()
        k = p.rhs()
        return _apply_inner(G, _radiation(G, stage, k)) if G.radiation else k

    def finish(s):
        if not G.radiation:  # post-update: enforce, extrapolate outward, parity, enforce
            s = _enforce_det(G, s)
            s = _apply_inner(G, _extrapolate(s[..., :-G.NG], G.NG, 3))
        return _enforce_det(G, s)

    k1 = slope(y)
    k2 = slope(finish(y + 0.5 * dt * k1))
    k3 = slope(finish(y + 0.5 * dt * k2))
    k4 = slope(finish(y + dt * k3))
    return finish(y + dt / 6 * k1 + dt / 3 * k2 + dt / 3 * k3 + dt / 6 * k4)


def _cfl_dt(G):
    xx, dxx = _grid(G, "cpu")
    r, drdx = _radius(G, xx[0])[:2]
    ds = [(drdx * dxx[0]).abs().min(), (r * dxx[1]).abs().min(),
          (r.abs().min() * torch.sin(xx[1]).abs().min() * dxx[2]).abs()]
    return G.CFL * float(min(ds))


def _wave_step(y, dt, inv):
    def slope(s):
        acc = 0
        for k in R3:
            off = [2, 2, 2]
            d = 0
            for o, w in _stencils(4)["dd"]:
                off[k] = 2 + o
                N = [n - 4 for n in s.shape[1:]]
                d = d + float(w) * s[0, off[2]:off[2] + N[0], off[1]:off[1] + N[1], off[0]:off[0] + N[2]]
            acc = acc + d * inv[k] ** 2
        return torch.stack([s[1, 2:-2, 2:-2, 2:-2], acc])

    def finish(s):
        # ghost layers from the inside out; the composition of the three directions does not
        # depend on their order, as each is the same linear map along its own axis
        for dim in (3, 2, 1):
            s = _extrapolate(s, 2, dim)
            s = _extrapolate(s.flip(dim), 2, dim).flip(dim)
        return s

    core = y[:, 2:-2, 2:-2, 2:-2]
    k1 = slope(y)
    k2 = slope(finish(core + 0.5 * dt * k1))
    k3 = slope(finish(core + 0.5 * dt * k2))
    k4 = slope(finish(core + dt * k3))
    return finish(core + dt / 6 * k1 + dt / 3 * k2 + dt / 3 * k3 + dt / 6 * k4)


@torch.no_grad()
def exact(case, seed, device="cuda"):
    kind = case["kind"]
    if kind == "wave":
        N = (case["N0"], case["N1"], case["N2"])
        y = _wave_initial(case, seed, device)
        dt = 0.5 * min(20.0 / n for n in N)
        for _ in range(case["steps"]):
            y = _wave_step(y, dt, [n / 20.0 for n in N])
        return y.unbind(0)
    if kind == "ensemble":  # the first three members: all of them take too long
        out = [None] * case["members"]
        for k, m in enumerate(_members(case)[:3]):
            G = _Build(m)
            out[k] = _initial(G, seed * 1009 + k, device)
            for _ in range(case["steps"]):
                out[k] = _step(G, out[k], _cfl_dt(G))
        return out
    G = _Build(case)
    y = _initial(G, seed, device)
    if kind == "diagnostics":
        return _exact_diagnostics(G, y)
    dt = _cfl_dt(G)
    if kind == "gradient":
        states = [y]
        for _ in range(case["steps"]):
            states.append(_step(G, states[-1], dt))
        lam = _cotangent(G, seed, device)
        for s in reversed(states[:-1]):
            with torch.enable_grad():
                s = s.clone().requires_grad_(True)
                (lam,) = torch.autograd.grad(_step(G, s, dt), s, lam)
        return {"y": states[-1].unbind(0), "gradient": lam.unbind(0)}
    for _ in range(case["steps"]):
        y = _step(G, y, dt)
    return y.unbind(0)


def _exact_diagnostics(G, y):
    M = _Metric(G, y.device, interior=True)
    p = _Point(G, M, y)
    p.ricci()
    c = p.constraints()
    dV = (M.s[0] * M.s[1] * M.s[2]).abs() * math.prod(M.dxx)
    shape = tuple(reversed(G.Nxx))
    integrals = {}
    for recipe in RECIPES:
        keep = (M.s[1] > 8.0 if recipe != RECIPES[0] else torch.ones_like(M.s[1], dtype=torch.bool)).expand(shape)
        w = torch.where(keep, dV.expand(shape), 0.0)
        vol = float(w.sum())
        d = {"volume": vol}
        for name, f in zip(INTEGRANDS, (c[0], c[4], c[5])):
            i = float((f * f * w).sum())
            d[name] = {"integral": i, "L2": math.sqrt(i), "RMS": math.sqrt(i / vol)}
        integrals[recipe] = d
    return {"fields": [torch.nn.functional.pad(f, (G.NG,) * 6) for f in c], "integrals": integrals}
