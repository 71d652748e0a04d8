"""The work that users of this solver have it do, as measurable cases.

A case is a dict of plain values.  prepare(case, seed) builds what a user's
program holds before it calls the solver (mesh, device context, state),
run(state) makes one pass through the public entry points of
sddc_amd.solver and returns everything the pass produced, work(case) gives
the bytes and operations the pass cannot do without, and exact(case, seed)
gives the same outputs from a plain double-precision PyTorch formulation of
the discretisation (no device library).

Kinds of pass:

  march      the time loop of the run driver: steps in blocks of ten with
             the residual norms of each block, then the state (or, with
             out="plot", the sensor and the nodal values of the Tecplot
             output) for the user's files
  stages     a host that drives the Runge-Kutta stages itself
  residual   a host program that keeps the state in its own arrays and has
             one residual evaluated per call (the Fortran drop-in's contract)
  ensemble   many independent runs stepped together (parameter studies)
  adjoint    forward run with checkpoints and the reverse pass of the wall
             drag (gradients for design and control)
  pullback   one vector-Jacobian product of the residual (implicit and
             matrix-free solvers)
"""
from __future__ import annotations

import dataclasses
import functools
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from sddc_amd import abi
from sddc_amd import cases as C
from sddc_amd import mesh as M
from sddc_amd import tecplot as TP
from sddc_amd.solver import Sd2d, Sd2dEnsemble

GAM = M.GAM
FREE = ("rinf", "pinf", "uinf", "vinf", "bxinf", "byinf")

# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
DEFAULTS = {"precision": "fp64", "k_stage": 3, "mu": 0.0, "eta0": 0.0, "out": "state", "nre": 1}


def _case(name, kind, mesh, nx, ny, N, **kw):
    c = {"kind": kind, "mesh": mesh, "nx": nx, "ny": ny, "N": N, **kw}
    return {"name": name, **c} if name else c


def listed():
    return [
        # a unit test or a coupled code: one step of a tiny channel with every
        # boundary type, the caller driving the five stages
        _case("tiny channel, host stages", "stages", "channel", 13, 9, 3),
        # the smallest cylinder run of the benchmark (32 x 64, p = 3)
        _case("cylinder 32x64 N4", "march", "ogrid", 32, 64, 4, steps=20),
        # a run that writes its Tecplot output (sensor and nodal values, NRE = 2)
        _case("vortex 131x62 N3 plot", "march", "periodic", 131, 62, 3, steps=10, out="plot", nre=2),
        # the headline benchmark (512 x 1024, p = 4)
        _case("cylinder 512x1024 N5", "march", "ogrid", 512, 1024, 5, steps=50),
        # the mixed-precision form on the periodic vortex (p = 3)
        _case("vortex 512x512 N4 mixed", "march", "periodic", 512, 512, 4, steps=50,
              precision="mixed"),
        # the other Runge-Kutta scheme, odd sizes
        _case("vortex 193x121 N5 rk4", "march", "periodic", 193, 121, 5, steps=20, k_stage=5),
        # a viscous and resistive run (channel with walls, unordered cells)
        _case("viscous channel 151x90 N4", "march", "channel", 151, 90, 4, steps=10, mu=1e-3,
              eta0=1e-3),
        # a viscous and resistive cylinder, p = 4
        _case("viscous cylinder 128x256 N5", "march", "ogrid", 128, 256, 5, steps=10, mu=1e-3,
              eta0=2e-3),
        # the drop-in residual call of a host program
        _case("residual 64x128 N5", "residual", "ogrid", 64, 128, 5),
        # a parameter study: sixteen cylinders of several sizes and orders
        _case("ensemble 16 members", "ensemble", "ogrid", 64, 128, 0, steps=20, members=16,
              draw=4),
        # the wall-drag gradient of the benchmark's 128 x 256 cylinder
        _case("adjoint 128x256 N4", "adjoint", "ogrid", 128, 256, 4, steps=20, ckpt=10),
        # one residual pullback, odd sizes
        _case("pullback 97x163 N5", "pullback", "curved", 97, 163, 5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["march"] * 6 + ["stages", "residual", "ensemble", "adjoint", "pullback"])
    N = rng.choice([3, 4, 5])
    if kind == "ensemble":
        return _case(None, kind, "ogrid", _log(rng, 16, 96), _log(rng, 32, 200), 0,
                     steps=rng.randint(5, 25), members=rng.randint(3, 18),
                     draw=rng.randint(10, 10 ** 6))
    if kind in ("adjoint", "pullback", "residual"):
        mesh = rng.choice(["ogrid", "curved"])
        hi = 200 if kind != "adjoint" else 120
        c = _case(None, kind, mesh, _log(rng, 6, hi), _log(rng, 24, 2 * hi), N)
        if kind == "adjoint":
            c.update(steps=rng.randint(5, 25), ckpt=rng.randint(3, 12))
        return c
    mesh = rng.choice(["ogrid", "periodic", "channel", "curved"])
    if kind == "stages":
        return _case(None, kind, mesh, _log(rng, 6, 60), _log(rng, 24, 120), N)
    big = 90 if mesh == "channel" else 240
    c = _case(None, kind, mesh, _log(rng, 8, big), _log(rng, 24, 2 * big), N,
              steps=rng.choice([5, 10, 20, 30]))
    style = rng.choice(["fp64", "fp64", "mixed", "rk4", "viscous", "viscous", "plot"])
    if style == "mixed":
        c["precision"] = "mixed"
    elif style == "rk4":
        c["k_stage"] = 5
    elif style == "viscous":
        c.update(mu=rng.choice([0.0, 1e-3, 2e-3]), eta0=rng.choice([1e-3, 2e-3]))
    elif style == "plot":
        # where the current does not vanish: elsewhere the sensor, a quotient
        # by its square, is rounding
        c.update(out="plot", nre=rng.randint(1, 3), mesh=rng.choice(["periodic", "channel"]))
        c["nx"] = min(c["nx"], 90)
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
RAMP = 2.0     # radii over which the cylinder runs' start rises from the wall
CFL = 0.1


@functools.lru_cache(maxsize=4)
def _base(mesh, nx, ny, N):
    """Mesh, set-up arrays, smooth start state and time step of a geometry
    (what every run of a study shares)."""
    p = M.RunParams(N=N)
    if mesh in ("ogrid", "curved"):
        m = M.ogrid(nx, ny, 0.5, 15.0, curved=mesh == "curved")
        p.curve_wall = int(mesh == "curved")
    elif mesh == "channel":
        m = M.channel(nx, ny, lx=0.2 * nx, ly=0.2 * ny, seed=nx, free_left=ny // 3)
    else:
        m = M.periodic_square(nx, ny)
        p = M.RunParams(N=N, dxcycl=m.dxcycl, dycycl=m.dycycl, rinf=25.0 / 9.0, pinf=5.0 / 3.0,
                        uinf=0.0, vinf=0.0, bxinf=0.0, byinf=0.0)
    case = M.build_case(m, p)
    if mesh in ("ogrid", "curved"):
        q = M.freestream_state(case, wall_ramp=(0.5, RAMP))
    elif mesh == "channel":
        q = M.smooth_perturbed_state(case, 0.05, seed=nx)
    else:
        q = M.orszag_tang_state(case, rho_pert=0.0)
    return case, q, C.cfl_dt(case, q, CFL)


def _state(q0, seed, amp=1e-3):
    """The start state of one run: density and velocity perturbed point by
    point at fixed pressure (and energy made consistent)."""
    t = q0.T                                    # (ncell, N, N, 9)
    rng = np.random.default_rng(seed)
    f = 1.0 + amp * rng.uniform(-1.0, 1.0, size=t.shape[:3])
    rho = t[..., 0] * f
    u = t[..., 1] / t[..., 0] + amp * rng.uniform(-1.0, 1.0, size=t.shape[:3])
    v = t[..., 2] / t[..., 0] + amp * rng.uniform(-1.0, 1.0, size=t.shape[:3])
    ke0 = 0.5 * (t[..., 1] ** 2 + t[..., 2] ** 2) / t[..., 0]
    out = np.array(t, order="C")
    out[..., 0] = rho
    out[..., 1] = rho * u
    out[..., 2] = rho * v
    out[..., 4] = t[..., 4] - ke0 + 0.5 * rho * (u * u + v * v)
    return out.T


def _inputs(case, seed):
    """(Case, start state) of a single-run case."""
    case = {**DEFAULTS, **case}
    base, q0, dt = _base(case["mesh"], case["nx"], case["ny"], case["N"])
    p = dataclasses.replace(base.params, dt=dt, k_stage=case["k_stage"], mu=case["mu"],
                            eta0=case["eta0"], nre=case["nre"])
    return dataclasses.replace(base, params=p), _state(q0, seed)


def _members(case, seed):
    """[(Case, start state)] of an ensemble: sizes, orders, Mach numbers and
    fields drawn from the case's own seed, perturbations from `seed`."""
    rng = np.random.default_rng(case["draw"])
    out = []
    for i in range(case["members"]):
        k = int(rng.integers(0, 3))
        N = int(rng.integers(3, 6))
        mach, ma, ang = rng.uniform(1.2, 2.0), rng.uniform(4.0, 8.0), rng.uniform(0.0, 90.0)
        nx, ny = max(4, case["nx"] >> k), max(12, case["ny"] >> k)
        base, q0 = _member_base(nx, ny, N, float(mach), float(ma), float(ang))
        out.append((base, _state(q0, seed + 1000 * i)))
    return out


@functools.lru_cache(maxsize=64)
def _member_base(nx, ny, N, mach, ma, ang):
    m, _, _ = _ensemble_mesh(nx, ny, N)
    bmag, th = mach / ma, math.radians(ang)
    p = dataclasses.replace(m.params, uinf=mach, bxinf=bmag * math.cos(th),
                            byinf=bmag * math.sin(th))
    case = dataclasses.replace(m, params=p)
    q = M.freestream_state(case, wall_ramp=(0.5, RAMP))
    p.dt = C.cfl_dt(case, q, CFL)
    return case, q


@functools.lru_cache(maxsize=16)
def _ensemble_mesh(nx, ny, N):
    return _base.__wrapped__("ogrid", nx, ny, N)


def _start(shape, seed, scale=1.0):
    return np.asfortranarray(scale * np.random.default_rng(seed).standard_normal(shape[::-1]).T)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        mem = _members(case, seed)
        e = Sd2dEnsemble([c for c, _ in mem])
        for i, (_, q) in enumerate(mem):
            e.set_state(i, q, [0.0, 0.0, 0.0, 0.0])
        return {"case": dict(case), "ens": e}
    case = {**DEFAULTS, **case}
    mc, q = _inputs(case, seed)
    prec = abi.SD2D_MIXED if case["precision"] == "mixed" else abi.SD2D_FP64
    g = Sd2d(mc, precision=prec)
    s = {"case": case, "g": g}
    g.set_state(q, [0.0, 0.0, 0.0, 0.0])
    if kind == "residual":
        s["q"] = q
    if kind == "pullback":
        g.compresid(want_resid=False, want_nabla=False)   # the lagged maxima
        s["rbar"] = _start(q.shape, seed + 7)
    if kind == "adjoint":
        s["qbar"] = _start(q.shape, seed + 7, 1e-3)
    if case["out"] == "plot":
        s["topo"] = TP.plot_topology(mc, case["nre"])
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ensemble":
        e = state["ens"]
        e.step(case["steps"])
        out = []
        for i in range(case["members"]):
            q, mx = e.get_state(i)
            out.append({"q": q, "maxima": mx})
        return out
    g = state["g"]
    if kind == "march":
        rows = []
        left = case["steps"]
        while left > 0:                      # the run driver's loop
            n = min(10, left)
            g.step(n, 10)
            d = g.diag()
            rows.append([d["ctime"], d["resid_rms"], d["divb_rms"], d["eigvmax_g"]])
            left -= n
        if case["out"] == "plot":
            sm, mu, eps = g.get_av()
            plotq, plotav = g.plot_nodes(state["topo"], mu)
            return {"rows": np.array(rows), "sensor": sm, "mu": mu, "eps": eps, "plotq": plotq,
                    "plotav": plotav}
        q, mx = g.get_state()
        return {"rows": np.array(rows), "q": q, "maxima": mx}
    if kind == "stages":
        for k in range(1, 6):
            g.rk_stage(k)
        q, mx = g.get_state()
        return {"q": q, "maxima": mx}
    if kind == "residual":
        g.set_state(state["q"])
        r, nabla = g.compresid()
        return {"resid": r, "nabla": nabla, "maxima": g.maxima()}
    if kind == "adjoint":
        J = g.fwd(case["steps"], case["ckpt"])
        q0b, pb, _ = g.vjp(state["qbar"], 1.0)
        return {"J": J, "qbar": q0b, "pbar": pb}
    q, ch, pb = g.compresid_vjp(state["rbar"])
    return {"qbar": q, "chbar": ch, "pbar": pb}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _march_bytes(N, k_stage, precision):
    """Per point and Runge-Kutta stage: the state passes of the scheme and
    the metrics, each once."""
    return C.alg_bytes_per_dof_stage(N, k_stage, 4 if precision == "mixed" else 8)


def work(case):
    case = {**DEFAULTS, **case}
    kind = case["kind"]
    if kind == "ensemble":
        rng = np.random.default_rng(case["draw"])
        by = fl = 0.0
        for _ in range(case["members"]):
            k, N = int(rng.integers(0, 3)), int(rng.integers(3, 6))
            rng.uniform(size=3)
            n = max(4, case["nx"] >> k) * max(12, case["ny"] >> k) * N * N
            by += n * (5 * case["steps"] * _march_bytes(N, 3, "fp64") + 72)
            fl += n * 5 * case["steps"] * 870.0
        return {"bytes": by, "flops": fl}
    N = case["N"]
    n = case["nx"] * case["ny"] * N * N
    metrics = 8 * (N * N + 4 * N * (N + 1)) / (N * N)
    stage = _march_bytes(N, case["k_stage"], case["precision"])
    flops = 870.0 + (1500.0 if case["mu"] or case["eta0"] else 0.0)
    if kind == "march":
        return {"bytes": n * (5 * case["steps"] * stage + 72), "flops": n * 5 * case["steps"] * flops}
    if kind == "stages":
        return {"bytes": n * (5 * stage + 72), "flops": n * 5 * flops}
    if kind == "residual":
        return {"bytes": n * (72 + 72 + 144 + metrics), "flops": n * 1400.0}
    pull = 3 * 72 + metrics                     # state, cotangent in and out
    if kind == "adjoint":
        ev = 5 * case["steps"]
        return {"bytes": n * (ev * (2 * stage + pull) + 2 * 72), "flops": n * ev * (2 * 870.0 + 2500.0)}
    return {"bytes": n * pull, "flops": n * 3000.0}


# ---------------------------------------------------------------------------
# the same in plain double-precision PyTorch
# ---------------------------------------------------------------------------
class _Geometry:
    """Operators, metrics and face lists of a case as tensors.  Fields are
    [v, i, j, cell]; face traces [local face, v, m, cell] with m the point
    number along the face as the cell itself walks it."""

    def __init__(self, case, dev):
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
        self.N, self.dev, p = case.N, dev, case.params
        self.L, self.Mm = t(case.lmat), t(case.mmat)
        self.jac = t(case.jac)
        self.s1, self.s2 = t(case.s1), t(case.s2)      # [a, b, rfp, js, c], [a, b, is, rfp, c]
        self.mu, self.eta0, self.alpha = p.mu, p.eta0, p.alpha
        self.par = {k: torch.tensor(float(getattr(p, k)), dtype=torch.float64, device=dev)
                    for k in FREE}
        f = np.asarray(case.topo.if2c, dtype=np.int64)
        it = f[np.asarray(case.topo.ibfinter, dtype=np.int64) - 1]
        pr = np.asarray(case.topo.cyc2fpair, dtype=np.int64).reshape(-1, 2) - 1
        two = np.concatenate([np.stack([it[:, 0], it[:, 2], it[:, 1], it[:, 3]], 1),
                              np.stack([f[pr[:, 0], 0], f[pr[:, 0], 2], f[pr[:, 1], 0],
                                        f[pr[:, 1], 2]], 1)]) - 1
        self.two = tuple(t(two[:, k]) for k in range(4))
        self.bnd = {}
        for typ, ids in case.topo.lists.items():
            if typ != "CYCL" and len(ids):
                b = f[np.asarray(ids, dtype=np.int64) - 1]
                self.bnd[typ] = (t(b[:, 0] - 1), t(b[:, 2] - 1))
        self.nc = case.ncell
        # normals at the face points, and the other family's metric there
        self.fn = self.faces(self.s1[0], self.s2[1])
        self.fo = self.faces(self.s1[1], self.s2[0])

    def faces(self, x, y):
        """Face-point values of x [v, r, j, c] and y [v, i, r, c]."""
        return torch.stack([y[:, :, 0], x[:, -1], y[:, :, -1].flip(1), x[:, 0].flip(1)])

    def with_ends(self, x, y, F):
        """x and y with their end flux points replaced by the faces'."""
        x = torch.cat([F[3].flip(1)[:, None], x[:, 1:-1], F[1][:, None]], 1)
        y = torch.cat([F[0][:, :, None], y[:, :, 1:-1], F[2].flip(1)[:, :, None]], 2)
        return x, y

    def traces(self, q):
        return torch.einsum("ri,vijc->vrjc", self.L, q), torch.einsum("rj,vijc->virc", self.L, q)

    def diff(self, x, y):
        return torch.einsum("ri,vrjc->vijc", self.Mm, x), torch.einsum("rj,virc->vijc", self.Mm, y)


def _pressure(q):
    return (GAM - 1.0) * (q[4] - 0.5 * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2) / q[0]
                          - 0.5 * (q[5] ** 2 + q[6] ** 2 + q[7] ** 2) - 0.5 * q[8] ** 2)


def _flux(q, ch, sx, sy):
    """Ideal-MHD and divergence-cleaning flux through the normal (sx, sy)."""
    u, v, w = q[1] / q[0], q[2] / q[0], q[3] / q[0]
    b2 = 0.5 * (q[5] ** 2 + q[6] ** 2 + q[7] ** 2)
    pt = _pressure(q) + b2
    un, bn = u * sx + v * sy, q[5] * sx + q[6] * sy
    e = q[4] - 0.5 * q[8] ** 2 + pt
    x = v * q[5] - u * q[6]
    return torch.stack([q[0] * un, q[1] * un + pt * sx - q[5] * bn, q[2] * un + pt * sy - q[6] * bn,
                        q[3] * un - q[7] * bn,
                        un * e - bn * (u * q[5] + v * q[6] + w * q[7]) + ch * q[8] * bn,
                        x * sy + ch * q[8] * sx, -x * sx + ch * q[8] * sy, q[7] * un - w * bn,
                        ch * bn])


def _speed(q):
    return torch.maximum(torch.maximum((q[1] / q[0]).abs(), (q[2] / q[0]).abs()),
                         (q[3] / q[0]).abs())


def _rusanov(ql, qr, sx, sy, ch):
    """Rusanov flux through the outward normal (sx, sy) of the left cell;
    the face's wave speed and velocity bound."""
    mag = torch.sqrt(sx ** 2 + sy ** 2)
    ux, uy = sx / mag, sy / mag
    vn = 0.5 * ((ql[1] * ux + ql[2] * uy) / ql[0] + (qr[1] * ux + qr[2] * uy) / qr[0])
    b = 0.5 * (ql[5:8] + qr[5:8])
    rs = ql[0] + qr[0]
    ca = GAM * (_pressure(ql) + _pressure(qr)) / rs
    cd = 2.0 * (b ** 2).sum(0) / rs
    cn = 2.0 * (b[0] * ux + b[1] * uy) ** 2 / rs
    ev = vn.abs() + torch.sqrt(0.5 * (ca + cd + torch.sqrt((ca + cd) ** 2 - 4.0 * ca * cn)))
    F = 0.5 * (_flux(ql, ch, sx, sy) + _flux(qr, ch, sx, sy) - mag * ev * (qr - ql))
    vel = 0.5 * (ql[1:4] / ql[0] + qr[1:4] / qr[0]).abs()
    return F, ev, vel.amax(0)


def _ghost(typ, q, nx, ny, p):
    one = torch.ones_like(q[0])
    psi2 = 0.5 * q[8] ** 2
    pe = p["pinf"] / (GAM - 1.0)
    bx, by = p["bxinf"] * one, p["byinf"] * one
    eb = 0.5 * (bx ** 2 + by ** 2)
    if typ == "INLE":
        r, u, v = p["rinf"] * one, p["uinf"], p["vinf"]
        return torch.stack([r, r * u, r * v, 0 * one, pe + 0.5 * r * (u * u + v * v) + eb + psi2, bx,
                            by, 0 * one, q[8]])
    if typ == "OUTL":
        return torch.stack([q[0], q[1], q[2], 0 * one,
                            pe + 0.5 * (q[1] ** 2 + q[2] ** 2) / q[0] + eb + psi2, bx, by, 0 * one,
                            0 * one])
    if typ == "WALL":
        return torch.stack([q[0], -q[1], -q[2], -q[3], q[4], -q[5], -q[6], -q[7], q[8]])
    if typ == "SYMP":
        r = 2.0 * p["rinf"] - q[0]
        n2 = nx ** 2 + ny ** 2
        un = (q[1] * nx + q[2] * ny) / (q[0] * n2)
        m1, m2, m3 = r * (q[1] / q[0] - 2 * un * nx), r * (q[2] / q[0] - 2 * un * ny), -r * q[3] / q[0]
        e = pe + 0.5 / r * (m1 ** 2 + m2 ** 2 + m3 ** 2) + eb + 0.5 * q[7] ** 2 + psi2
        return torch.stack([r, m1, m2, m3, e, bx, by, -q[7], q[8]])
    return q.clone()


def _residual(G, q, ch):
    """resid and nablaQs of q for the cleaning speed ch, and the largest
    wave speed and velocity bound of the evaluation."""
    tx, ty = G.traces(q)
    ux, uy = G.s1[0], G.s2[1]
    FT = G.faces(tx, ty)
    FF, FQ = torch.zeros_like(FT), torch.zeros_like(FT)
    pick = lambda A, k, c: A[k, :, :, c].permute(1, 2, 0)   # noqa: E731  [v, m, face]

    def put(A, k, c, x):                                    # the inverse of pick
        x = x.permute(2, 0, 1)
        return A.permute(0, 3, 1, 2).index_put((k, c), x).permute(0, 2, 3, 1)

    out = lambda k, one: torch.where((k == 0) | (k == 3), -one, one)   # noqa: E731
    one = torch.ones((), dtype=torch.float64, device=G.dev)
    eig, um = [], [_speed(tx[:, 1:-1]).amax(), _speed(ty[:, :, 1:-1]).amax()]
    cl, kl, cr, kr = G.two
    if len(cl):
        ql, qr = pick(FT, kl, cl), pick(FT, kr, cr).flip(1)
        n = out(kl, one) * pick(G.fn, kl, cl)
        F, e, u = _rusanov(ql, qr, n[0], n[1], ch)
        a = 0.5 * (ql + qr)
        FF = put(put(FF, kl, cl, out(kl, one) * F), kr, cr, -out(kr, one) * F.flip(1))
        FQ = put(put(FQ, kl, cl, a), kr, cr, a.flip(1))
        eig.append(e.amax())
        um.append(u.amax())
    for typ, (c, k) in G.bnd.items():
        ql = pick(FT, k, c)
        n = out(k, one) * pick(G.fn, k, c)
        qr = _ghost(typ, ql, n[0], n[1], G.par)
        F, e, u = _rusanov(ql, qr, n[0], n[1], ch)
        FF = put(FF, k, c, out(k, one) * F)
        FQ = put(FQ, k, c, 0.5 * (ql + qr))
        eig.append(e.amax())
        um.append(u.amax())
    fx, fy = G.with_ends(_flux(tx, ch, ux[0], ux[1]), _flux(ty, ch, uy[0], uy[1]), FF)
    ax, ay = G.with_ends(tx, ty, FQ)
    nabla = torch.stack([sum(G.diff(ax * ux[d], ay * uy[d])) / G.jac for d in (0, 1)], 1)
    dx, dy = G.diff(fx, fy)
    D = dx + dy
    if G.mu or G.eta0:
        D = D - _viscous(G, q, ax, ay, FT, FQ, nabla, pick, put)
    r = list((-D / G.jac).unbind(0))
    divb = nabla[5, 0] + nabla[6, 1]
    u, v, w = q[1] / q[0], q[2] / q[0], q[3] / q[0]
    src = [None, q[5], q[6], q[7], u * q[5] + v * q[6] + w * q[7], u, v, w, None]
    for k in range(1, 8):
        r[k] = r[k] - divb * src[k]
    r[8] = r[8] - G.alpha * q[8]
    return torch.stack(r), nabla, torch.stack(eig).amax(), torch.stack(um).amax()


def _viscous(G, q, ax, ay, FT, FQ, nabla, pick, put):
    """Divergence of the viscous and resistive fluxes (BR1)."""
    g = nabla.reshape(18, *nabla.shape[2:])            # [v*2 + d]
    gx, gy = G.traces(g)
    GT = G.faces(gx, gy)
    GF = GT.clone()
    cl, kl, cr, kr = G.two
    if len(cl):
        a = 0.5 * (pick(GT, kl, cl) + pick(GT, kr, cr).flip(1))
        GF = put(put(GF, kl, cl, a), kr, cr, a.flip(1))
    if "WALL" in G.bnd:
        c, k = G.bnd["WALL"]
        e = lambda s: (s[4] - 0.5 * (s[1] ** 2 + s[2] ** 2 + s[3] ** 2) / s[0]  # noqa: E731
                       - 0.5 * (s[5:9] ** 2).sum(0)) / s[0]
        ex, ey = G.diff(e(ax)[None], e(ay)[None])      # along xi and eta
        # the derivative across the wall's own family, traced to the face
        DE = G.faces(G.traces(ey)[0], G.traces(ex)[1])
        qo, gl = pick(FT, k, c), pick(GT, k, c)
        de, o = pick(DE, k, c)[0], pick(G.fo, k, c)
        u, v, w = qo[1] / qo[0], qo[2] / qo[0], qo[3] / qo[0]
        ei, k2 = e(qo), u * u + v * v + w * w
        gx_ = gl[0::2]                                 # d/dx of the nine variables
        dbp = (qo[5:9] * gx_[5:9]).sum(0)
        gr = gl.clone()
        for d in (0, 1):
            h = gl[d::2]
            dke = 0.5 * k2 * h[0] + u * (h[1] - u * h[0]) + v * (h[2] - v * h[0]) + w * (h[3] - w * h[0])
            gr[8 + d] = -h[4] + 2.0 * ei * h[0] + 2.0 * dke + dbp + 2.0 * de * o[d] * qo[0]
        GF = put(GF, k, c, 0.5 * (gl + gr))
    gx, gy = G.with_ends(gx, gy, GF)
    fx = _vflux(ax, gx, G.mu, G.eta0, G.s1[0][0], G.s1[0][1])
    fy = _vflux(ay, gy, G.mu, G.eta0, G.s2[1][0], G.s2[1][1])
    dx, dy = G.diff(fx, fy)
    return dx + dy


def _vflux(q, g, mu, eta, sx, sy):
    u, v, w = q[1] / q[0], q[2] / q[0], q[3] / q[0]
    k2 = u * u + v * v + w * w
    ei = (q[4] - 0.5 * k2 * q[0] - 0.5 * (q[5:9] ** 2).sum(0)) / q[0]
    d = [g[0::2], g[1::2]]
    du, dv, dw, de = [], [], [], []
    for h in d:
        du.append((h[1] - h[0] * u) / q[0])
        dv.append((h[2] - h[0] * v) / q[0])
        dw.append((h[3] - h[0] * w) / q[0])
        dke = 0.5 * k2 * h[0] + q[0] * (u * du[-1] + v * dv[-1] + w * dw[-1])
        de.append((h[4] - dke - (q[5:9] * h[5:9]).sum(0) - h[0] * ei) / q[0])
    div = du[0] + dv[1]
    sh, k = dv[0] + du[1], GAM / 0.72
    txx, tyy = mu * (2.0 * du[0] - 2.0 / 3.0 * div), mu * (2.0 * dv[1] - 2.0 / 3.0 * div)
    jx, jy, jz = d[1][7], -d[0][7], d[0][6] - d[1][5]
    F4 = u * txx + v * mu * sh + w * mu * dw[0] + mu * k * de[0] + eta * (jz * q[6] - jy * q[7])
    G4 = u * mu * sh + v * tyy + w * mu * dw[1] + mu * k * de[1] + eta * (jx * q[7] - jz * q[5])
    z = torch.zeros_like(u)
    return torch.stack([z, txx * sx + mu * sh * sy, mu * sh * sx + tyy * sy,
                        mu * (dw[0] * sx + dw[1] * sy), F4 * sx + G4 * sy, -eta * jz * sy,
                        eta * jz * sx, eta * (jx * sy - jy * sx), z])


def _sensor(case, q, nabla):
    """SM_IND of the artificial viscosity."""
    _, lo, hi = M.av_projectors(case.N)
    f = torch.from_numpy(hi @ lo).to(q)
    out = []
    for x in (q[0], (nabla[6, 0] - nabla[5, 1]) ** 2):
        s = torch.einsum("ai,bj,ijc->abc", f, f, x)
        out.append(torch.log10(((s - x) ** 2 / x ** 2).sum((0, 1))))
    return torch.stack(out)


S5P3 = ((1.0, 0.0, 0, 0.377268915331368), (1.0, 0.0, 0, 0.377268915331368),
        (0.644090224936674, 0.355909775063327, 0, 0.242995220537396),
        (0.632066208361863, 0.367933791638137, 0, 0.238458932846290),
        (0.762406163401431, 0.237593836598569, 2, 0.287632146308408))


class _Run:
    """State, running maxima and time of one run."""

    def __init__(self, G, case, q, mx=None):
        z = torch.zeros((), dtype=torch.float64, device=G.dev)
        self.G, self.case, self.q = G, case, q
        self.E, self.U = (z, z) if mx is None else mx
        self.t, self.it, self.last = 0.0, 0, None

    def resid(self, q):
        r, nabla, e, u = _residual(self.G, q, torch.sqrt((self.E * (self.E - self.U)).clamp_min(0))
                                   if float(self.E) > 0 else torch.zeros_like(self.E))
        self.E, self.U = torch.maximum(self.E, e), torch.maximum(self.U, u)
        self.last = (q, r, nabla)
        return r

    def step(self):
        dt, q0 = self.case.params.dt, self.q
        if self.case.params.k_stage == 3:
            qs = [q0]
            for a, b, k, c in S5P3:
                q = a * qs[-1] + c * dt * self.resid(qs[-1])
                qs.append(q + b * qs[k] if b else q)
            self.q = qs[-1]
        else:
            q1 = q0 + 0.39175222700392 * dt * self.resid(q0)
            q2 = 0.44437049406734 * q0 + 0.55562950593266 * q1 + 0.36841059262959 * dt * self.resid(q1)
            q3 = 0.6201018513854 * q0 + 0.3798981486146 * q2 + 0.25189177424738 * dt * self.resid(q2)
            r3 = self.resid(q3)
            q4 = 0.17807995410773 * q0 + 0.82192004589227 * q3 + 0.54497475021237 * dt * r3
            self.q = (0.00683325884039 * q0 + 0.51723167208978 * q2 + 0.12759831133288 * q3
                      + 0.34833675773694 * q4
                      + dt * (0.08460416338212 * r3 + 0.22600748319395 * self.resid(q4)))
        self.t += dt
        self.it += 1

    def norms(self):
        _, r, nabla = self.last
        n = nabla[0, 0].numel()
        return (math.sqrt(float((r ** 2).sum()) / (9 * n)),
                math.sqrt(float(((nabla[5, 0] + nabla[6, 1]) ** 2).sum()) / n))

    def maxima(self):
        return np.array([float(self.E), float(self.U), float(self.E), float(self.U)])


def _host(t):
    return np.asfortranarray(t.detach().cpu().numpy())


def _plot(case, q, topo, mu):
    """Nodal averages of the cells' solution polynomials, as primitives."""
    N, n1 = case.N, topo.nre + 1
    h = torch.tensor([[M._lagrange(case.xs, i, k / topo.nre) for i in range(N)] for k in range(n1)],
                     dtype=torch.float64, device=q.device)
    val = torch.einsum("ai,bj,vijc->vcba", h, h, q).reshape(9, -1)      # cell*(n1^2) + ii + n1*jj
    cnt = torch.from_numpy(np.diff(topo.xadj).astype(np.int64)).to(q.device)
    node = torch.repeat_interleave(torch.arange(topo.nnode, device=q.device), cnt)
    occ = torch.from_numpy(topo.contrib.astype(np.int64)).to(q.device)
    a = torch.zeros(9, topo.nnode, dtype=torch.float64, device=q.device)
    a = a.index_add(1, node, val[:, occ]) / cnt
    m = torch.zeros(2, topo.nnode, dtype=torch.float64, device=q.device)
    m = m.index_add(1, node, torch.from_numpy(np.ascontiguousarray(mu)).to(q)[:, occ // (n1 * n1)]) / cnt
    u, v, w = a[1] / a[0], a[2] / a[0], a[3] / a[0]
    p = (GAM - 1) * (a[4] - 0.5 * a[0] * (u * u + v * v + w * w)
                     - 0.5 * (a[5] ** 2 + a[6] ** 2 + a[7] ** 2))
    return _host(torch.stack([a[0], u, v, w, p, a[5], a[6], a[7], a[8]])), _host(m)


def _mu_av(case, sm, E):
    p, N = case.params, case.N
    eps = E * math.sqrt(p.dxcycl * p.dycycl / case.ncell) / (N - 1) * 0.05
    lo, hi = np.array([[-5.0], [-3.0]]), np.array([[0.0], [1.0]])
    mid = eps / 2 * (1 + np.sin(np.pi * (sm - (lo + hi) / 2) / (hi - lo)))
    return np.where(sm < lo, 0.0, np.where(sm > hi, eps, mid)), eps


def _drag(G, case, q):
    """Wall drag: pressure times the outward normal's x component."""
    xs, N = case.xs, case.N
    w = []
    for i in range(N):
        c = np.poly1d([1.0])
        for j in range(N):
            if j != i:
                c = c * np.poly1d([1.0, -xs[j]]) / (xs[i] - xs[j])
        w.append(float(np.polyint(c)(1.0)))
    c, k = G.bnd["WALL"]
    t = G.faces(*G.traces(q))[k, :, :, c].permute(1, 2, 0)
    n = G.fn[k, :, :, c].permute(1, 2, 0)[0] * torch.where((k == 0) | (k == 3), -1.0, 1.0)
    wt = torch.tensor(w, dtype=torch.float64, device=q.device)[:, None]
    # the weights are symmetric under the reversal of a face's direction
    return (wt * _pressure(t) * n).sum()


def _evaluations(case):
    return {"march": 5, "stages": 5, "ensemble": 5, "adjoint": 30}.get(case["kind"], 3) * case.get("steps", 1)


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if case["kind"] == "ensemble":
        out = []
        for mc, q in _members(case, seed):
            with torch.no_grad():
                R = _Run(_Geometry(mc, dev), mc, torch.from_numpy(q).to(dev).contiguous())
                for _ in range(case["steps"]):
                    R.step()
            out.append({"q": _host(R.q), "maxima": R.maxima()})
        return out
    case = {**DEFAULTS, **case}
    if case["nx"] * case["ny"] * case["N"] ** 2 * _evaluations(case) > 3.4e9:
        return None
    mc, q = _inputs(case, seed)
    G = _Geometry(mc, dev)
    q = torch.from_numpy(q).to(dev).contiguous()
    kind = case["kind"]
    if kind == "adjoint":
        return _exact_adjoint(G, mc, q, case, seed)
    if kind == "pullback":
        with torch.no_grad():
            R = _Run(G, mc, q)
            R.resid(q)
            ch = torch.sqrt(R.E * (R.E - R.U))
        x = q.clone().requires_grad_()
        ch.requires_grad_()
        G.par = {k: v.requires_grad_() for k, v in G.par.items()}
        rbar = torch.from_numpy(_start(tuple(q.shape), seed + 7)).to(dev)
        g = torch.autograd.grad((_residual(G, x, ch)[0] * rbar).sum(),
                                [x, ch] + [G.par[k] for k in FREE], allow_unused=True)
        pb = np.array([0.0 if v is None else float(v) for v in g[2:]])
        return {"qbar": _host(g[0]), "chbar": float(g[1]), "pbar": pb}
    with torch.no_grad():
        R = _Run(G, mc, q)
        if kind == "residual":
            r = R.resid(q)
            return {"resid": _host(r), "nabla": _host(R.last[2]), "maxima": R.maxima()}
        if kind == "stages":
            R.step()
            return {"q": _host(R.q), "maxima": R.maxima()}
        rows, left, nrm = [], case["steps"], (0.0, 0.0)
        while left > 0:
            n = min(10, left)
            for _ in range(n):
                R.step()
                if R.it % 10 == 1:
                    nrm = R.norms()
            rows.append([R.t, nrm[0], nrm[1], float(R.E)])
            left -= n
        if case["out"] == "plot":
            sm = _host(_sensor(mc, R.last[0], R.last[2]))
            mu, eps = _mu_av(mc, sm, float(R.E))
            pq, pav = _plot(mc, R.q, TP.plot_topology(mc, case["nre"]), mu)
            return {"rows": np.array(rows), "sensor": sm, "mu": mu, "eps": eps, "plotq": pq,
                    "plotav": pav}
        return {"rows": np.array(rows), "q": _host(R.q), "maxima": R.maxima()}


def _exact_adjoint(G, mc, q, case, seed):
    """J, and the cotangents of the start state and the free stream, by
    automatic differentiation of the stepping above (one step at a time
    recomputed in the backward pass)."""
    x = q.clone().requires_grad_()
    G.par = {k: v.requires_grad_() for k, v in G.par.items()}

    def one(q, E, U, *par):
        H = object.__new__(_Geometry)
        H.__dict__.update(G.__dict__, par=dict(zip(FREE, par)))
        R = _Run(H, mc, q, (E, U))
        R.step()
        return R.q, R.E, R.U, _drag(H, mc, R.q)

    z = torch.zeros((), dtype=torch.float64, device=q.device)
    cur, E, U, J = x, z, z, z
    for _ in range(case["steps"]):
        cur, E, U, d = checkpoint(one, cur, E, U, *[G.par[k] for k in FREE], use_reentrant=False)
        J = J + d / case["steps"]
    qbar = torch.from_numpy(_start(tuple(q.shape), seed + 7, 1e-3)).to(q.device)
    g = torch.autograd.grad(J + (cur * qbar).sum(), [x] + [G.par[k] for k in FREE],
                            allow_unused=True)
    pb = np.array([0.0 if v is None else float(v) for v in g[1:]])
    return {"J": float(J), "qbar": _host(g[0]), "pbar": pb}
