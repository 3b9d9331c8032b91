"""Performance cases: the runs that a user of this framework has it do, through its public
entry points (DGSEM, LSRK54, ARK23, LSRKEnsemble), on states of the kind they meet.

Kinds (a pass is `steps` time steps of a run in progress, its state staying on the device):

  vortex    2-D Euler isentropic vortex, periodic, entropy-conservative flux differencing + Rusanov, LSRK54
  bubble    3-D Euler-with-gravity warm bubble, walls, entropy-conservative flux differencing + Roe, LSRK54
  sw        2-D shallow water, periodic, weak form + Rusanov, LSRK54
  ensemble  many shallow-water instances of uneven size and degree, one launch per stage
  wave      density wave of the Euler or advection law in 1 to 3 dimensions, weak form + Rusanov, LSRK54
  imex      Euler with gravity, horizontally explicit, vertically implicit, ARK23

`precision` is the operator's own option: "reference" (its default: the reference's summation order) or "fast".
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "atum.jl_amd"))
import atum_hip as A  # noqa: E402
from atum_hip import _lib  # noqa: E402

GAMMA, GRAV, CV_D, T_REF, P_S = 1.4, 9.81, 719.0, 300.0, 1e5
R_D = GAMMA * CV_D - CV_D
GM1 = GAMMA - 1


# ---- the cases ----------------------------------------------------------------
def listed():
    return [
        # the smallest run: one step at a time, as solve_ with an after_step hook takes them
        {"name": "vortex_8_n4_step", "kind": "vortex", "K": 8, "N": 4, "steps": 1, "precision": "reference"},
        # a served vortex request: odd mesh, high degree
        {"name": "vortex_45_n6_fast", "kind": "vortex", "K": 45, "N": 6, "steps": 2, "precision": "fast"},
        # the framework's headline configuration
        {"name": "bubble_16_n4_fast", "kind": "bubble", "K": 16, "N": 4, "steps": 2, "precision": "fast"},
        # a large single run, whose stage exceeds the last-level cache
        {"name": "bubble_24_n4_fast", "kind": "bubble", "K": 24, "N": 4, "steps": 2, "precision": "fast"},
        # the highest degree, few large elements
        {"name": "bubble_9_n7_fast", "kind": "bubble", "K": 9, "N": 7, "steps": 2, "precision": "fast"},
        # the same physics in the operator's default arithmetic
        {"name": "bubble_12_n4_reference", "kind": "bubble", "K": 12, "N": 4, "steps": 2, "precision": "reference"},
        # one large weak-form run
        {"name": "sw_256_n3", "kind": "sw", "K": 256, "N": 3, "steps": 2},
        # an ensemble study: uneven meshes and degrees
        {"name": "ensemble_40", "kind": "ensemble", "members": 40, "kmax": 64, "steps": 2},
        # convergence studies of the plain weak form
        {"name": "wave_euler_3d_20_n4", "kind": "wave", "law": "euler", "dim": 3, "K": 20, "N": 4, "steps": 2},
        {"name": "wave_advection_2d_80_n4", "kind": "wave", "law": "advection", "dim": 2, "K": 80, "N": 4,
         "steps": 2},
        # atmosphere columns, horizontally explicit and vertically implicit: the benchmark's mesh, a small odd one
        {"name": "imex_32x10_n3_fast", "kind": "imex", "K": 32, "KV": 10, "N": 3, "steps": 2, "precision": "fast"},
        {"name": "imex_11x7_n3_reference", "kind": "imex", "K": 11, "KV": 7, "N": 3, "steps": 2,
         "precision": "reference"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: the degrees 3 to 7 of the workloads (1 to 7 for the bubble and the waves),
    meshes from a few elements to about 8 million unknowns (1.2 million in reference arithmetic)."""
    kind = rng.choices(["vortex", "bubble", "sw", "ensemble", "wave", "imex"], [5, 5, 3, 2, 3, 2])[0]
    precision = rng.choice(["fast", "reference"])
    most = 8.0e6 if precision == "fast" else 1.2e6
    if kind == "vortex":
        n = rng.randint(3, 7)
        k = _log_int(rng, 8, min(128, int(math.sqrt(most / 4) / (n + 1))))
        return {"kind": kind, "K": k, "N": n, "steps": rng.choice([1, 2]), "precision": precision}
    if kind == "bubble":
        n = rng.randint(1, 7)
        k = _log_int(rng, 3, min(40, int((most / 5) ** (1 / 3) / (n + 1))))
        return {"kind": kind, "K": k, "N": n, "steps": 2, "precision": precision}
    if kind == "sw":
        n = rng.randint(3, 7)
        return {"kind": kind, "K": _log_int(rng, 8, min(256, int(1400 / (n + 1)))), "N": n, "steps": 2}
    if kind == "ensemble":
        return {"kind": kind, "members": rng.randint(6, 40), "kmax": rng.randint(16, 64), "steps": 2}
    if kind == "wave":
        law, dim, n = rng.choice(["euler", "advection"]), rng.randint(1, 3), rng.randint(1, 7)
        top = {1: 2000, 2: int(500 / (n + 1)), 3: int(90 / (n + 1))}[dim]
        return {"kind": kind, "law": law, "dim": dim, "K": _log_int(rng, 4, top), "N": n, "steps": 2}
    return {"kind": kind, "K": rng.randint(8, 32 if precision == "fast" else 20), "KV": rng.randint(6, 10), "N": 3,
            "steps": rng.choice([1, 2]), "precision": precision}


# ---- meshes and states ----------------------------------------------------------
def _members(case, seed):
    """The ensemble's members (K, N): the same meshes for every seed, another state for each."""
    rng = np.random.Generator(np.random.PCG64(20260101 + case["members"] + 1000 * case["kmax"]))
    return [{"kind": "sw", "K": int(rng.integers(8, case["kmax"] + 1)), "N": int(rng.integers(3, 8)),
             "seed": seed * 1000 + i} for i in range(case["members"])]


def _coords(case):
    k = case["K"]
    if case["kind"] == "vortex":
        return [np.linspace(-5, 5, k + 1)] * 2, (True, True)
    if case["kind"] == "bubble":
        return [np.linspace(0, 2000, k + 1)] * 3, (False,) * 3
    if case["kind"] == "sw":
        return [np.linspace(0, 1, k + 1)] * 2, (True, True)
    if case["kind"] == "wave":
        return [np.linspace(-1, 1, k + 1)] * case["dim"], (True,) * case["dim"]
    x, z = np.linspace(0, 20e3, k + 1), np.linspace(0, 10e3, case["KV"] + 1)
    return [x, x, z], (True, True, False)


def _grid(case):
    coords, periodic = _coords(case)
    order = "stacked" if case["kind"] == "imex" else "cartesian"
    return A.brickgrid(A.LobattoCell(case["N"], len(coords)), coords, periodic, order, lazy=True)


def _isothermal(z):
    rho = P_S / (T_REF * R_D) * np.exp(-GRAV / (R_D * T_REF) * z)
    return rho, rho * R_D * T_REF


def _warm(x, theta1):
    """State at rest on the isothermal background with potential temperature theta1 added at fixed pressure."""
    rho0, p = _isothermal(x[-1])
    exner = (p / P_S) ** (R_D / (GAMMA * CV_D))
    t = (p / (rho0 * R_D) / exner + theta1) * exner
    rho, zero = p / (R_D * t), np.zeros_like(p)
    return np.stack([rho, zero, zero, zero, rho * (CV_D * t + GRAV * x[-1])])


def _state(case, x, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    if case["kind"] == "vortex":
        c, beta = rng.uniform(-2, 2, 2), rng.uniform(4, 5.5)
        r0, r1 = x[0] - c[0], x[1] - c[1]
        f = beta * np.exp(1 - (r0 * r0 + r1 * r1))
        rho = (1 - GM1 * f ** 2 / (16 * GAMMA * np.pi ** 2)) ** (1 / GM1)
        u, v, p = 1 - f / (2 * np.pi) * r1, 1 + f / (2 * np.pi) * r0, rho ** GAMMA
        return np.stack([rho, rho * u, rho * v, p / GM1 + rho * (u * u + v * v) / 2])
    if case["kind"] == "bubble":
        c = np.array([1000.0, 1000.0, 350.0]) + rng.uniform(-100, 100, 3)
        r2 = sum((x[d] - c[d]) ** 2 for d in range(3))
        return _warm(x, rng.uniform(1.5, 2.5) * np.exp(-r2 / 250.0 ** 2))
    if case["kind"] == "sw":
        a, w, c = rng.uniform(0.01, 0.1), rng.uniform(0.05, 0.2), rng.uniform(0, 1, 2)
        h = 1 + a * np.exp(-((x[0] - c[0]) ** 2 + (x[1] - c[1]) ** 2) / w ** 2)
        zero = np.zeros_like(h)
        return np.stack([h, zero, zero, h * rng.uniform(0, 1)])
    if case["kind"] == "wave":
        rho = 2 + rng.uniform(0.5, 1) * np.sin(np.pi * (x.sum(axis=0) - rng.uniform(0, 2)))
        if case["law"] == "advection":
            return rho[None, :]
        return np.stack([rho] + [rho] * case["dim"] + [1 / GM1 + case["dim"] * rho / 2])
    return _warm(x, 0.1 * rng.standard_normal(x.shape[1]))


def _dt(case, grid):
    h = float(np.min(np.diff(grid.coords[0])))
    n = case["N"]
    if case["kind"] == "vortex":
        return 0.1 * h / n
    if case["kind"] == "bubble":
        return (0.25 if n < 5 else 0.125) * h / n / 330.0
    if case["kind"] == "sw":
        return 0.125 * h / n / math.sqrt(GRAV * 1.1)
    if case["kind"] == "wave":
        return 0.25 * h / n / case["dim"] / math.sqrt(GAMMA)
    return 0.2 * grid.min_node_distance(dims=(0, 1)) / 330.0


def _operator(case, grid):
    kind = case["kind"]
    ec = A.FluxDifferencingForm(A.EntropyConservativeFlux())
    if kind == "vortex":
        return A.DGSEM(law=A.EulerLaw(2), grid=grid, volume_form=ec, surface_numericalflux=A.RusanovFlux(),
                       precision=case["precision"], geometry="device")
    if kind == "bubble":
        law = A.EulerGravityLaw(3, grav=GRAV, problem=A.Problem(boundary="reflect"))
        return A.DGSEM(law=law, grid=grid, volume_form=ec, surface_numericalflux=A.RoeFlux(),
                       precision=case["precision"], geometry="device")
    if kind == "sw":
        return A.DGSEM(law=A.ShallowWaterLaw(2, grav=GRAV), grid=grid, surface_numericalflux=A.RusanovFlux(),
                       geometry="device")
    if kind == "wave":
        law = A.EulerLaw(case["dim"]) if case["law"] == "euler" else A.AdvectionLaw(case["dim"])
        return A.DGSEM(law=law, grid=grid, surface_numericalflux=A.RusanovFlux(), geometry="device")
    prob = A.Problem(boundary="reflect", referencestate=lambda x: _isothermal(x[-1]))
    law = A.EulerGravityLaw(3, grav=GRAV, problem=prob)
    ex = A.DGSEM(law=law, grid=grid, volume_form=ec, surface_numericalflux=A.RusanovFlux(),
                 precision=case["precision"], geometry="device")
    lin = A.DGSEM(law=A.LinearEulerGravityLaw(law), grid=grid, surface_numericalflux=A.RusanovFlux(),
                  directions=(3,), auxstate=ex.auxstate, geometry="device")
    return ex, lin


class TensorField(A.Field):
    """A field over the memory of a torch tensor (Ns, Np*K), which stays the tensor's."""

    def __init__(self, tensor, ctx):
        self.ctx, self.tensor = ctx, tensor
        self.shape, self.nbytes = tuple(tensor.shape), tensor.numel() * 8
        self.ptr = _lib.c_void_p(tensor.data_ptr())

    def __del__(self):
        pass


def _field(q0, ctx):
    t = torch.from_numpy(q0).cuda()
    torch.cuda.synchronize()  # the framework's stream is its own
    return TensorField(t, ctx)


def prepare(case, seed):
    if case["kind"] == "ensemble":
        members = _members(case, seed)
        grids = [_grid(m) for m in members]
        dgs = [_operator(m, g) for m, g in zip(members, grids)]
        qs = [_field(_state(m, g.points, m["seed"]), d.ctx) for m, g, d in zip(members, grids, dgs)]
        solver = A.LSRKEnsemble(dgs, qs, [_dt(m, g) for m, g in zip(members, grids)])
        return {"ensemble": True, "solver": solver, "q": qs, "steps": case["steps"]}
    grid = _grid(case)
    op = _operator(case, grid)
    dt = _dt(case, grid)
    q0 = _state(case, grid.points, seed)
    if case["kind"] == "imex":
        ex, lin = op
        q = _field(q0, ex.ctx)
        solver = A.ARK23(ex, lin, q, dt, split_rhs=False)
    else:
        q = _field(q0, op.ctx)
        solver = A.LSRK54(op, q, dt)
    return {"ensemble": False, "solver": solver, "q": q, "steps": case["steps"]}


def run(state):
    if state["ensemble"]:
        state["solver"].run(state["steps"])
        return [q.tensor for q in state["q"]]
    if state["steps"] == 1:
        state["solver"].dostep(state["q"])
    else:
        state["solver"].run(state["q"], state["steps"])
    return state["q"].tensor


# ---- what a pass cannot do without -----------------------------------------------
def _stage_work(case):
    """Of one stage: the state read and the new one written, the solver's dq read and written (each stage needs
    its neighbours' previous one, so nothing shorter than a stage moves less), geopotential and reference
    state; operations of the volume term (each unordered pair of a line once) and of the faces."""
    kind, nq = case["kind"], case["N"] + 1
    dim = {"vortex": 2, "bubble": 3, "sw": 2, "wave": case.get("dim"), "imex": 3}[kind]
    ns = 1 if case.get("law") == "advection" else dim + 2
    nodes = (case["K"] ** 2 * case["KV"] if kind == "imex" else case["K"] ** dim) * nq ** dim
    nbytes = nodes * 8.0 * (4 * ns + {"bubble": 1, "imex": 3}.get(kind, 0))
    if kind in ("vortex", "bubble", "imex"):
        flops = nodes * dim * (nq - 1) / 2 * (50 + 10 * ns)
    else:
        flops = nodes * dim * (2 * ns * nq + 4 * ns)
    flops += nodes * dim * 2 / nq * (12 * ns)
    return nbytes, flops, nodes


def work(case):
    if case["kind"] == "ensemble":
        w = [work(dict(m, steps=case["steps"])) for m in _members(case, 0)]
        return {"bytes": sum(v["bytes"] for v in w), "flops": sum(v["flops"] for v in w)}
    nbytes, flops, nodes = _stage_work(case)
    stages = 5 * case["steps"]
    if case["kind"] == "imex":
        # three explicit and three linear tendencies, two banded solves (block form: four products of
        # half-filled blocks of 5 Nq rows for every block of a line)
        stages = 3 * case["steps"]
        nbytes += nodes * 8.0 * 2 * 5 * 2 / 3
        flops += nodes * (2 * 5 * 4 + 40) + nodes * 5 * 4 * (5 * (case["N"] + 1)) * 2 / 3
    return {"bytes": nbytes * stages, "flops": flops * stages}


# ---- the same steps in plain torch, 64 bits ----------------------------------------
class _Brick:
    """Fields as (components, [Kz,] [Ky,] Kx, [nz,] [ny,] nx) on a brick of rectangular elements."""

    def __init__(self, case):
        self.case = case
        coords, self.periodic = _coords(case)
        self.dim, self.nq = len(coords), case["N"] + 1
        cell = A.LobattoCell(case["N"], 1)
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.D, self.w = self.t(cell.D), self.t(cell.weights_1d)
        self.kd = [len(c) - 1 for c in coords]
        self.h = [self.t(np.diff(c)) for c in coords]
        x = []
        xi = cell.points_1d
        for d, c in enumerate(coords):
            p = self.t((1 - xi)[None, :] / 2 * c[:-1, None] + (1 + xi)[None, :] / 2 * c[1:, None])
            x.append(self.along(p, d))
        self.x = x
        self.stacked = case["kind"] == "imex"

    def t(self, a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(self.dev)

    def along(self, p, d):
        """An array over (elements, nodes) of direction d, shaped to broadcast over a field."""
        shape = [1] * (2 * self.dim)
        shape[self.dim - 1 - d], shape[2 * self.dim - 1 - d] = p.shape[0], p.shape[1]
        return p.reshape(shape)

    def field(self, q):
        n = [self.nq] * self.dim
        if not self.stacked:
            return q.reshape([q.shape[0]] + self.kd[::-1] + n)
        kx, ky, kz = self.kd
        return q.reshape([q.shape[0], ky, kx, kz] + n).permute(0, 3, 1, 2, 4, 5, 6)

    def flat(self, f):
        if self.stacked:
            f = f.permute(0, 2, 3, 1, 4, 5, 6)
        return f.reshape(f.shape[0], -1)

    def axes(self, r):
        """Element and node axis of direction r in a field."""
        return self.dim - r, 2 * self.dim - r

    def hr(self, r):
        """2/h of direction r, shaped to broadcast over a field's components."""
        return self.along((2 / self.h[r])[:, None], r)

    def ends(self, f, r):
        """The values at the low and high end of direction r, and the neighbours' there."""
        e, n = self.axes(r)
        lo, hi = f.select(n, 0), f.select(n, self.nq - 1)
        return lo, hi, hi.roll(1, e), lo.roll(-1, e)

    def wall(self, r, side):
        """Which of the elements' low (0) or high (1) faces in direction r are on a wall."""
        m = torch.zeros(self.kd[r], dtype=torch.bool, device=self.dev)
        m[0 if side == 0 else -1] = not self.periodic[r]
        shape = [1] * (2 * self.dim - 1)
        shape[self.dim - 1 - r] = self.kd[r]
        return m.reshape(shape)

    def lift(self, dq, r, nf_lo, nf_hi):
        _, n = self.axes(r)
        c = self.hr(r).select(n - 1, 0)
        dq.select(n, 0).sub_(c * nf_lo / self.w[0])
        dq.select(n, self.nq - 1).sub_(c * nf_hi / self.w[-1])

    def weak(self, f, r):
        """Weak-form volume term of the flux component f in direction r."""
        _, n = self.axes(r)
        m = self.D * self.w[:, None] / self.w[None, :]  # [n, i]
        return self.hr(r) * torch.movedim(torch.tensordot(f, m, dims=([n], [0])), -1, n)


def _pressure(q, phi):
    ke = sum(q[1 + d] ** 2 for d in range(q.shape[0] - 2)) / (2 * q[0])
    return GM1 * (q[-1] - ke - q[0] * phi)


def _logmean(a, b):
    z = a / b
    f = (z - 1) / (z + 1)
    u = f * f
    series = 1 + u * (1 / 3 + u * (1 / 5 + u * (1 / 7 + u / 9)))
    far = u > 1e-4
    exact = torch.log(torch.where(far, z, torch.full_like(z, 2.0))) / (2 * torch.where(far, f, torch.ones_like(f)))
    return (a + b) / (2 * torch.where(far, exact, series))


def _euler_flux(q, a, r):
    p = _pressure(q, a[0])
    u = q[1 + r] / q[0]
    rows = [q[1 + r]] + [q[1 + d] * u + (p if d == r else 0) for d in range(q.shape[0] - 2)] + [u * (q[-1] + p)]
    return torch.stack(rows)


def _ec_volume(g, q, phi, r):
    """Flux differencing with the entropy-conservative flux along direction r (zero geopotential: no gravity)."""
    dim = g.dim
    _, n = g.axes(r)
    u = [q[1 + d] / q[0] for d in range(dim)]
    b = q[0] / (2 * _pressure(q, phi))
    m = g.D * (g.w[:, None] / g.w[None, :])  # [n, i]
    out = torch.zeros_like(q)
    for i in range(g.nq):
        for k in range(g.nq):
            if i == k:
                continue

            def at(v, j):
                return v.select(n - 1, j)

            r1, r2, b1, b2 = at(q[0], i), at(q[0], k), at(b, i), at(b, k)
            ua = [(at(v, i) + at(v, k)) / 2 for v in u]
            u2 = sum((at(v, i) ** 2 + at(v, k) ** 2) / 2 for v in u)
            rl, bl = _logmean(r1, r2), _logmean(b1, b2)
            fr = ua[r] * rl
            pd = (r1 + r2) / (2 * (b1 + b2))
            fu = [ua[d] * fr + (pd if d == r else 0) for d in range(dim)]
            f1, f2 = at(phi, i), at(phi, k)
            fe = (1 / (2 * GM1 * bl) - u2 / 2 + (f1 + f2) / 2) * fr + sum(x * y for x, y in zip(fu, ua))
            fu[r] = fu[r] - (b1 + b2) / 2 * rl / (2 * b1) * (f1 - f2)
            c = m[k, i] - g.D[i, k]
            out.select(n, i).add_(c * torch.stack([fr] + fu + [fe]))
    return g.hr(r) * out


def _roe(qm, qp, a, n, r):
    """Roe flux with normal n e_r, n = +-1 (the geopotential is continuous)."""
    dim, phi = qm.shape[0] - 2, a[0]
    pm, pp = _pressure(qm, phi), _pressure(qp, phi)
    um, up = qm[1:-1] / qm[0], qp[1:-1] / qp[0]
    sm, sp = qm[0].sqrt(), qp[0].sqrt()

    def mean(a, b):
        return (sm * a + sp * b) / (sm + sp)

    u = mean(um, up)
    h = mean((qm[-1] + pm) / qm[0], (qp[-1] + pp) / qp[0])
    c = mean((GAMMA * pm / qm[0]).sqrt(), (GAMMA * pp / qp[0]).sqrt())
    rho, un, du, dr, dp = sm * sp, n * u[r], up - um, qp[0] - qm[0], pp - pm
    dun = n * du[r]
    w1 = (un - c).abs() * (dp - rho * c * dun) / (2 * c * c)
    w2 = (un + c).abs() * (dp + rho * c * dun) / (2 * c * c)
    w3 = un.abs() * (dr - dp / (c * c))
    w4 = un.abs() * rho
    e = torch.zeros_like(u)
    e[r] = n
    fp = [(w1 + w2 + w3) / 2]
    fp += [(w1 * (u[d] - c * e[d]) + w2 * (u[d] + c * e[d]) + w3 * u[d] + w4 * (du[d] - dun * e[d])) / 2
           for d in range(dim)]
    fp.append((w1 * (h - c * un) + w2 * (h + c * un) + w3 * ((u * u).sum(0) / 2 + phi)
               + w4 * ((u * du).sum(0) - un * dun)) / 2)
    return n * (_euler_flux(qm, a, r) + _euler_flux(qp, a, r)) / 2 - torch.stack(fp)


def _rusanov(flux, speed, qm, am, qp, ap, n, r):
    ws = torch.maximum(speed(qm, am, r), speed(qp, ap, r))
    return n * (flux(qm, am, r) + flux(qp, ap, r)) / 2 - ws * (qp - qm) / 2


def _sound(q, a, r):
    return (q[1 + r] / q[0]).abs() + (GAMMA * _pressure(q, a[0]) / q[0]).sqrt()


def _sw_flux(q, _, r):
    u, p = q[1 + r] / q[0], GRAV * q[0] ** 2 / 2
    return torch.stack([q[1 + r]] + [q[1 + r] * (q[1 + d] / q[0]) + (p if d == r else 0) for d in range(2)] + [u * q[3]])


def _sw_speed(q, _, r):
    return (q[1 + r] / q[0]).abs() + (GRAV * q[0]).sqrt()


def _lin_flux(q, a, r):
    phi, ref_rho, ref_p = a
    p = GM1 * (q[-1] - q[0] * phi)
    h = (ref_p / GM1 + ref_rho * phi + ref_p) / ref_rho
    zero = torch.zeros_like(p)
    return torch.stack([q[1 + r]] + [p if d == r else zero for d in range(3)] + [h * q[1 + r]])


def _lin_speed(q, a, r):
    return (GAMMA * a[2] / a[1]).sqrt()


def _tendency(g, q, aux, flux, speed, directions, surface="rusanov", volume="weak"):
    dq = torch.zeros_like(q)
    for r in directions:
        dq += g.weak(flux(q, aux, r), r) if volume == "weak" else _ec_volume(g, q, aux[0], r)
        states = g.ends(q, r)
        auxes = list(zip(*[[v[0] for v in g.ends(a[None], r)] for a in aux])) or [()] * 4
        nf = []
        for side, n in ((0, -1.0), (1, 1.0)):
            m, p, am, ap = states[side], states[2 + side], auxes[side], auxes[2 + side]
            if not g.periodic[r]:
                wall = g.wall(r, side)
                mirror = m.clone()
                mirror[1 + r] = -m[1 + r]
                p = torch.where(wall, mirror, p)
                ap = tuple(torch.where(wall, y, x) for x, y in zip(ap, am))
            nf.append(_roe(m, p, am, n, r) if surface == "roe" else _rusanov(flux, speed, m, am, p, ap, n, r))
        g.lift(dq, r, *nf)
    return dq


_LSRK_A = (0.0, -567301805773 / 1357537059087, -2404267990393 / 2016746695238,
           -3550918686646 / 2091501179385, -1275806237668 / 842570457699)
_LSRK_B = (1432997174477 / 9575080441755, 5161836677717 / 13612068292357, 1720146321549 / 2090206949498,
           3134564353537 / 4481467310338, 2277821191437 / 14882151754819)


def _lsrk(rhs, q, dt, steps):
    dq = torch.zeros_like(q)
    for _ in range(steps):
        for a, b in zip(_LSRK_A, _LSRK_B):
            dq = a * dq + rhs(q)
            q = q + b * dt * dq
    return q


def _line_solver(g, lin, scale):
    """x -> (I + scale L)^-1 x for the vertical linear operator, whose matrix is the same in every column."""
    n = 5 * g.nq * g.kd[2]
    probe = torch.zeros([5, g.kd[2], 1, 1] + [g.nq] * 3, dtype=torch.float64, device=g.dev)
    cols = []
    for j in range(n):
        probe.zero_()
        ez, rem = divmod(j, 5 * g.nq)
        k, s = divmod(rem, 5)
        probe[s, ez, 0, 0, k] = 1
        cols.append(lin(probe)[:, :, 0, 0, :, 0, 0].permute(1, 2, 0).reshape(-1))
    lu = torch.linalg.lu_factor(torch.eye(n, dtype=torch.float64, device=g.dev) + scale * torch.stack(cols, dim=1))

    def solve(b):
        shape = b.shape
        v = b.permute(1, 4, 0, 2, 3, 5, 6).reshape(n, -1)
        x = torch.linalg.lu_solve(*lu, v).reshape(shape[1], g.nq, 5, shape[2], shape[3], g.nq, g.nq)
        return x.permute(2, 0, 3, 4, 1, 5, 6).contiguous()

    return solve


def _ark(ex, lin, solve, q, dt, steps):
    s2 = math.sqrt(2.0)
    ea = [[0, 0], [2 - s2, 0], [0.5, 0.5]]
    ia = [[0, 0], [1 - 1 / s2, 0], [1 / (2 * s2), 1 / (2 * s2)]]
    b = [1 / (2 * s2), 1 / (2 * s2), 1 - 1 / s2]
    for _ in range(steps):
        stage, ks = q, []
        for i in range(3):
            if i > 0:
                stage = solve(q + dt * sum(ea[i][k] * ks[k][0] + ia[i][k] * ks[k][1] for k in range(i)))
            im = lin(stage)
            ks.append((ex(stage) - im, im))
        q = q + dt * sum(b[k] * (ks[k][0] + ks[k][1]) for k in range(3))
    return q


def exact(case, seed):
    if case["kind"] == "ensemble":
        return [exact(dict(m, steps=case["steps"]), m["seed"]) for m in _members(case, seed)]
    grid = _grid(case)
    g = _Brick(case)
    dt = _dt(case, grid)
    q = g.field(g.t(_state(case, grid.points, seed))).contiguous()
    dirs = range(g.dim)
    kind = case["kind"]
    zero = torch.zeros_like(q[0])
    phi = (GRAV * g.x[-1]).expand(q.shape[1:])
    if kind == "vortex":
        args = ((zero,), _euler_flux, _sound, dirs, "rusanov", "ec")
    elif kind == "bubble":
        args = ((phi,), _euler_flux, _sound, dirs, "roe", "ec")
    elif kind == "sw":
        args = ((), _sw_flux, _sw_speed, dirs)
    elif kind == "wave" and case["law"] == "euler":
        args = ((zero,), _euler_flux, _sound, dirs)
    elif kind == "wave":
        args = ((), lambda p, a, r: p, lambda p, a, r: torch.ones_like(p[0]), dirs)
    else:
        aux = [GRAV * g.x[2]] + [g.t(v) for v in _isothermal(g.x[2].cpu().numpy())]

        def lin(v):
            out = _tendency(g, v, tuple(a.expand(v.shape[1:]) for a in aux), _lin_flux, _lin_speed, (2,))
            out[3] -= v[0] * GRAV
            return out

        solve = _line_solver(g, lin, -dt * (1 - 1 / math.sqrt(2)))
        return g.flat(_ark(lambda v: _tendency(g, v, (phi,), _euler_flux, _sound, dirs, volume="ec"), lin, solve, q,
                           dt, case["steps"]))
    return g.flat(_lsrk(lambda v: _tendency(g, v, *args), q, dt, case["steps"]))
