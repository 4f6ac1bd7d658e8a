"""Measured workloads of the gfx950 DG residual and SSP-RK3 step.

Each case is one thing that a program built on this package has the GPU do,
through the public classes (`SolverClass`, `Batch`):

  residual  one evaluation of R(U) with its monitoring data, and R read back
            (a steady-state check, a linearisation, a unit test)
  steps     a save interval: a number of synchronization steps, then the
            state read back (the reference's time loop with "Save solution
            every")
  batch     the same for many independent cases stepped together

over the polynomial degrees 2 to 6 with their integration rules, Cartesian and
curvilinear grids, FP64 and mixed precision, subgrid scale models and the open
box with characteristic boundaries, sponge and matching layer. The flow of
every case (phase shifts, Mach and Reynolds number, vortex and pulse centres)
is drawn from the seed.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from vcp3d_open_amd.cases import BATCH_RULE, OpenBoxCase, TGVCase
from vcp3d_open_amd.solver import Batch, SolverClass

GAMMA = 1.4
RK = ((1.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0))   # weights of U0 and dt R per stage


# ------------------------------------------------------------------- cases
def _tgv(mode, n, p, *, rule=0, curvilinear=False, precision="fp64", sgs="none", steps=0):
    return dict(mode=mode, flow="tgv", n=n, p=p, rule=rule or BATCH_RULE[p], curvilinear=curvilinear,
                precision=precision, sgs=sgs, steps=steps)


def _box(nx, ny, nz, p, *, sponge, inflow="static", precision="fp64", sgs="none", steps=1):
    return dict(mode="steps", flow="box", nx=nx, ny=ny, nz=nz, p=p, rule=BATCH_RULE[p], sponge=sponge,
                inflow=inflow, precision=precision, sgs=sgs, steps=steps)


def _many(count, n_low, n_high, *, precision="fp64", steps=1):
    return dict(mode="batch", flow="tgv", count=count, n_low=n_low, n_high=n_high, precision=precision, steps=steps)


def listed():
    return [
        # the smallest call: launches and the readback are most of it
        dict(_tgv("residual", 4, 2), name="residual_n4_p2"),
        # a small residual at a high degree, odd element count
        dict(_tgv("residual", 5, 5, curvilinear=True), name="residual_n5_p5_curv"),
        # the small case that the whole reference runs in its tests: 8^3, P = 3
        dict(_tgv("steps", 8, 3, steps=50), name="steps_n8_p3"),
        # low degree with an eddy-viscosity model
        dict(_tgv("steps", 18, 2, sgs="wale", steps=30), name="steps_n18_p2_wale"),
        # the integration rule that the reference's own P = 3 decks use
        dict(_tgv("steps", 14, 3, rule=10, curvilinear=True, steps=30), name="steps_n14_p3_rule10"),
        # a mid-size curvilinear case at the usual degree
        dict(_tgv("steps", 16, 4, curvilinear=True, steps=20), name="steps_n16_p4_curv"),
        # high degrees
        dict(_tgv("steps", 16, 5, curvilinear=True, steps=15), name="steps_n16_p5_curv"),
        dict(_tgv("steps", 11, 6, curvilinear=True, steps=10), name="steps_n11_p6_curv"),
        # the headline case: 32^3, P = 4, curvilinear, FP64
        dict(_tgv("steps", 32, 4, curvilinear=True, steps=30), name="steps_n32_p4_curv"),
        # the mixed-precision form
        dict(_tgv("steps", 20, 4, curvilinear=True, precision="mixed", steps=30), name="steps_n20_p4_mixed"),
        # PC-NSCBC in- and outflow, sponge and matching layer
        dict(_box(48, 24, 24, 4, sponge=8, steps=20), name="box_48x24x24_p4"),
        # independent cases of uneven degree and size stepped together
        dict(_many(16, 4, 13, steps=10), name="batch_16_cases"),
    ]


def _dofs(case):
    if case["flow"] == "box":
        return case["nx"] * case["ny"] * case["nz"] * (case["p"] + 1) ** 3
    return case["n"] ** 3 * (case["p"] + 1) ** 3


def draw(rng):
    def log_uniform(a, b):
        return math.exp(rng.uniform(math.log(a), math.log(b)))

    kind = rng.choice(["residual", "steps", "steps", "steps", "box", "batch"])
    precision = rng.choice(["fp64", "fp64", "fp64", "mixed"])
    if kind == "batch":
        low = rng.randint(3, 6)
        return _many(rng.randint(2, 14), low, low + rng.randint(2, 7), precision=precision, steps=rng.randint(3, 10))
    p = rng.randint(2, 6)
    # elements per direction: up to 1.7 million solution points, and for a
    # bare residual, whose readback would be most of it, up to 60 thousand
    top = ((6.0e4 if kind == "residual" else 1.7e6) ** (1.0 / 3.0)) / (p + 1)
    if kind == "box":
        ny, nz = int(log_uniform(2, 0.8 * top)), int(log_uniform(2, 0.8 * top))
        nx = int(log_uniform(4, 1.5 * top))
        return _box(nx, ny, nz, p, sponge=max(1, nx // 6), inflow=rng.choice(["static", "total"]),
                    precision=precision, sgs=rng.choice(["none", "none", "vreman"]), steps=rng.randint(5, 15))
    n = max(3, int(round(log_uniform(3, top))))
    curv = n >= 4 and rng.random() < 0.5
    rule = 10 if p == 3 and rng.random() < 0.5 else 0
    if kind == "residual":
        return _tgv("residual", n, p, rule=rule, curvilinear=curv)
    return _tgv("steps", n, p, rule=rule, curvilinear=curv, precision=precision,
                sgs=rng.choice(["none", "none", "wale", "vreman"]), steps=rng.randint(5, 25))


# ------------------------------------------------------------------ inputs
def _flows(case, seed):
    """The case objects that the seed gives: one, or one per batch member."""
    rng = np.random.default_rng([seed, 77])
    if case["flow"] == "box":
        return [OpenBoxCase(n=(case["nx"], case["ny"], case["nz"]), lengths=(2.0, 1.0, 1.0), p=case["p"],
                            rule=case["rule"], mach=float(rng.uniform(0.3, 0.7)), sponge_elems=case["sponge"],
                            inflow=case["inflow"], sgs=case["sgs"], seed=int(rng.integers(1 << 30)))]

    def flow():
        return dict(mach=float(rng.uniform(0.05, 0.4)),
                    reynolds=float(math.exp(rng.uniform(math.log(400.0), math.log(3200.0)))),
                    phase=tuple(float(x) for x in rng.uniform(0.0, 2.0 * math.pi, 3)))

    if case["mode"] == "batch":
        # the degrees and sizes belong to the case, the flows to the seed
        shape = random.Random(case["count"] * 1000 + case["n_low"] * 100 + case["n_high"])
        out = []
        for i in range(case["count"]):
            p, n = 2 + i % 5, shape.randint(case["n_low"], case["n_high"])
            out.append(TGVCase(n=n, p=p, rule=BATCH_RULE[p], **flow()))
        return out
    return [TGVCase(n=case["n"], p=case["p"], rule=case["rule"], curvilinear=case["curvilinear"], sgs=case["sgs"],
                    **flow())]


def prepare(case, seed):
    solvers = []
    for flow in _flows(case, seed):
        s = SolverClass(flow, precision=case.get("precision", "fp64"))
        s.ReadRestartSolution(flow.initial_conservative())
        if case["flow"] == "box":
            s.SetDampingState(flow.damping_primitive())
        solvers.append(s)
    state = dict(mode=case["mode"], steps=case.get("steps", 0), solvers=solvers,
                 precision=case.get("precision", "fp64"))
    if case["mode"] == "batch":
        state["batch"] = Batch()
        for s in solvers:
            state["batch"].add(s)
    return state


def _saved(state, array):
    """An array as the program keeps it. The mixed form evaluates the residual
    in single precision: its results are kept in that."""
    return torch.from_numpy(array).to(torch.float32) if state["precision"] == "mixed" else array


def run(state):
    solvers = state["solvers"]
    if state["mode"] == "residual":
        monitoring = solvers[0].Residual(True)
        return dict(residual=solvers[0].residual_array(), monitoring=monitoring)
    if state["mode"] == "batch":
        state["batch"].step(state["steps"])
        state["batch"].wait()
        return dict(solution=[_saved(state, s.solution()) for s in solvers])
    rk_steps = 0
    for _ in range(state["steps"]):
        monitoring = solvers[0].ExecuteTimeSynchronizationStep()
        rk_steps += solvers[0].last_rk_steps
    return dict(solution=_saved(state, solvers[0].solution()), monitoring=_saved(state, monitoring),
                rk_steps=rk_steps)


# -------------------------------------------------------------------- work
def _residual_work(n_elem, p, rule):
    """Bytes and flops of one residual evaluation: per element the state, the
    volume and face metric terms and the residual, FP64; sum-factorised
    contractions (2 flops per multiply-add), 350 flops per integration point
    and 700 per face point of pointwise physics, four iterations of the
    mass-matrix solve."""
    K, M = p + 1, rule // 2 + 1
    fwd = 5 * (2 * K ** 3 * M + 3 * K * K * M * M + 4 * K * M ** 3)
    bwd = 5 * (3 * K * M ** 3 + 3 * K * K * M * M + 2 * K ** 3 * M)
    solve = 10 * (K ** 3 * M + K * K * M * M + K * M ** 3) + 30 * M ** 3 + 55 * K ** 3
    face = 10 * (2 * K ** 3 + 3 * K * K * M + 4 * K * M * M) + 10 * (4 * K * M * M + 3 * K * K * M)
    flops = 2.0 * (fwd + bwd + 4 * solve + 3 * face) + 350.0 * M ** 3 + 3 * 700.0 * M * M
    bytes_ = 8.0 * (10 * K ** 3 + 10 * M ** 3 + 3 * 22 * M * M + 16)
    return n_elem * bytes_, n_elem * flops


def work(case):
    bytes_ = flops = 0.0
    for flow in _flows(case, 0):
        n = 1 if case["mode"] == "residual" else 3 * case["steps"]
        b, f = _residual_work(flow.n_elems, flow.p, flow.rule)
        if case["mode"] != "residual":   # two of three stages read the step's state too
            b += flow.n_elems * 8.0 * 5 * flow.n_dofs * 2.0 / 3.0
        bytes_ += n * b
        flops += n * f
    return dict(bytes=bytes_, flops=flops)


# ------------------------------------------- the same in plain torch, 64 bits
class _Plain:
    """The scheme of a periodic Taylor-Green case in dense tensor algebra:
    entropy variables in the orthonormal Legendre basis, Gauss integration,
    Ismail-Roe and viscous fluxes with penalty and symmetrising terms, and the
    mass matrix dU/dV solved to rounding. Arrays are [element][...][k][j][i]
    with the elements in their [nk][nj][ni] order."""

    def __init__(self, flow):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.flow, self.K, self.M = flow, flow.p + 1, flow.rule // 2 + 1
        self.E, self.n = flow.n_elems, flow.n_elem[::-1]
        self.mu = flow.ref["mu_nondim"]
        leg = np.polynomial.legendre
        r, w = leg.leggauss(self.M)
        ends = np.array([-1.0, 1.0])
        # grid and solution nodes: Legendre-Gauss-Lobatto
        inner = np.sort(leg.legroots(leg.legder([0.0] * flow.p + [1.0]))) if flow.p > 1 else np.zeros(0)
        for _ in range(3):
            d = leg.Legendre([0.0] * flow.p + [1.0]).deriv()
            inner = inner - d(inner) / d.deriv()(inner)
        nodes = np.concatenate([[-1.0], inner, [1.0]])

        def basis(x, deriv):
            cols = []
            for q in range(self.K):
                c = leg.Legendre([0.0] * q + [math.sqrt(q + 0.5)])
                cols.append((c.deriv() if deriv else c)(x) + 0.0 * x)
            return np.stack(cols, axis=1)

        inv = np.linalg.inv(basis(nodes, False))
        f64 = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=self.dev)
        self.A, self.D = f64(basis(r, False)), f64(basis(r, True))          # [point][mode]
        self.F, self.dF = f64(basis(ends, False)), f64(basis(ends, True))   # [side][mode]
        lag = lambda x, deriv: f64(basis(x, deriv) @ inv)                   # [point][node]
        L, dL, Lf, dLf = lag(r, False), lag(r, True), lag(ends, False), lag(ends, True)
        self.LN, self.dLN, self.VI = f64(basis(nodes, False)), f64(basis(nodes, True)), f64(inv)
        w = f64(w)
        self.w2 = w[:, None] * w[None, :]
        self.w3 = w[:, None, None] * self.w2
        X = f64(flow.element_grid()).reshape(self.E, 3, self.K, self.K, self.K)
        cols = [self._to(X, *o) for o in ((dL, L, L), (L, dL, L), (L, L, dL))]
        self.J, self.m = self._metric(*cols)
        vol = (self.w3 * self.J).sum((1, 2, 3))
        self.les = vol ** (1.0 / 3.0) / flow.p
        # faces: normal along +d and area factor, inverse metric, per side
        self.fn, self.fa, self.fm, self.length = [], [], [], []
        for d in range(3):
            nrm, area, met = [], [], []
            for s in range(2):
                ops = []
                for a in range(3):
                    o = [L, L, L]
                    o[d] = Lf[s:s + 1]
                    o[a] = dLf[s:s + 1] if a == d else dL
                    ops.append(self._to(X, *o).reshape(self.E, 3, self.M, self.M))
                n = torch.linalg.cross(ops[(d + 1) % 3], ops[(d + 2) % 3], dim=1)
                a = n.norm(dim=1)
                nrm.append(n / a[:, None]); area.append(a); met.append(self._metric(*ops)[1])
            self.fn.append(nrm); self.fa.append(area); self.fm.append(met)
            self.length.append(2.0 * vol / sum((self.w2 * a).sum((1, 2)) for a in area))
        self.dt = flow.dt_synchr * flow.ref["u_ref"]

    @staticmethod
    def _to(x, ox, oy, oz):
        """Operators along i, j and k of [..., k, j, i]."""
        x = torch.matmul(x, ox.T)
        x = torch.matmul(oy, x)
        return torch.matmul(oz, x.flatten(-2)).unflatten(-1, (oy.shape[0], ox.shape[0]))

    @staticmethod
    def _back(x, ox, oy, oz):
        return _Plain._to(x, ox.T.contiguous(), oy.T.contiguous(), oz.T.contiguous())

    @staticmethod
    def _metric(dr, ds, dt):
        J = (dr * torch.linalg.cross(ds, dt, dim=1)).sum(1)
        m = torch.stack([torch.linalg.cross(ds, dt, dim=1), torch.linalg.cross(dt, dr, dim=1),
                         torch.linalg.cross(dr, ds, dim=1)], 1) / J[:, None, None]
        return J, m                                                          # m[e][r s t][x y z][points]

    def start(self):
        """Modal entropy variables of the initial state."""
        q = torch.tensor(self.flow.initial_conservative(), dtype=torch.float64, device=self.dev)
        ref = self.flow.ref
        rho, vel = q[..., 0], q[..., 1:4] / q[..., 0:1]
        p = 0.4 * (q[..., 4] - 0.5 * rho * (vel * vel).sum(-1)) / ref["p_ref"]
        rho, vel = rho / ref["rho_ref"], vel / ref["u_ref"]
        s = torch.log(p / rho ** GAMMA)
        V = [(GAMMA - s) / 0.4 - 0.5 * rho * (vel * vel).sum(-1) / p]
        V += [rho * vel[..., i] / p for i in range(3)] + [-rho / p]
        V = torch.stack(V, 1).reshape(self.E, 5, self.K, self.K, self.K)
        return self._to(V, self.VI, self.VI, self.VI)

    @staticmethod
    def _primitive(V):
        vel = -V[:, 1:4] / V[:, 4:5]
        ek = 0.5 * (vel * vel).sum(1)
        rho = (-V[:, 4] * torch.exp(GAMMA - 0.4 * (V[:, 0] - V[:, 4] * ek))) ** -2.5
        return rho, vel, -rho / V[:, 4], ek

    def _cartesian(self, G, m):
        """Parametric derivatives G[r s t] of the five variables to Cartesian
        ones, variable l with the metric of integration point l, which is what
        the default (reference-compatible) mode does."""
        c = m.flatten(3)[:, :, :, :5]                                        # [e][r s t][x y z][l]
        pad = (slice(None), slice(None)) + (None,) * (G[0].dim() - 2)
        return [sum(G[r] * c[:, r, x][pad] for r in range(3)) for x in range(3)]

    def _eddy(self, rho, G, length):
        """Eddy viscosity of the case's model; G[i][j] = du_i / dx_j."""
        G = torch.stack([torch.stack(row, -1) for row in G], -2)
        tr = lambda a: (a.diagonal(dim1=-2, dim2=-1).sum(-1) / 3.0)[..., None, None] * torch.eye(
            3, dtype=a.dtype, device=a.device)
        sq = lambda a: (a * a).sum((-2, -1))
        length = length.reshape((-1,) + (1,) * (rho.dim() - 1))
        if self.flow.sgs == "wale":
            S, G2 = 0.5 * (G + G.mT), torch.matmul(G, G)
            Sd = 0.5 * (G2 + G2.mT) - tr(G2)
            den = sq(S) ** 2.5 + sq(Sd) ** 1.25
            return rho * (0.325 * length) ** 2 * sq(Sd) ** 1.5 / den.clamp_min(1e-30)
        al = G - tr(G)
        be = length[..., None, None] ** 2 * torch.matmul(al, al.mT.contiguous())
        B = sum(be[..., i, i] * be[..., j, j] - be[..., i, j] ** 2 for i, j in ((0, 1), (0, 2), (1, 2)))
        return rho * 0.07 * (B.clamp_min(0.0) / sq(al).clamp_min(1e-30)).sqrt()

    def _viscous(self, V4, vel, G, mu, ev):
        """Stress tensor and heat flux from the Cartesian entropy gradients."""
        iv = 1.0 / V4
        du = [[-iv * (G[x][:, 1 + i] + vel[:, i] * G[x][:, 4]) for x in range(3)] for i in range(3)]
        div = -2.0 / 3.0 * (du[0][0] + du[1][1] + du[2][2])
        tau = [[(mu + ev) * (du[i][j] + du[j][i] + (div if i == j else 0.0)) for j in range(3)] for i in range(3)]
        k = mu * GAMMA / 0.72 + ev * GAMMA / 0.9
        q = [-k * iv * iv / 0.4 * G[x][:, 4] for x in range(3)]
        return du, tau, q

    def _volume(self, U):
        A, D = self.A, self.D
        V = self._to(U, A, A, A)
        G = self._cartesian([self._to(U, D, A, A), self._to(U, A, D, A), self._to(U, A, A, D)], self.m)
        rho, vel, p, ek = self._primitive(V)
        ev = torch.zeros_like(rho)
        du, tau, q = self._viscous(V[:, 4], vel, G, self.mu, ev)
        if self.flow.sgs != "none":
            ev = self._eddy(rho, du, self.les)
            du, tau, q = self._viscous(V[:, 4], vel, G, self.mu, ev)
        E = p / 0.4 + rho * ek
        wJ = self.w3 * self.J
        res = 0.0
        cart = []
        for x in range(3):
            f = [rho * vel[:, x]] + [rho * vel[:, x] * vel[:, i] - tau[i][x] + (p if i == x else 0.0) for i in range(3)]
            f.append((E + p) * vel[:, x] - sum(vel[:, i] * tau[i][x] for i in range(3)) + q[x])
            cart.append(torch.stack(f, 1))
        for d, o in enumerate(((D, A, A), (A, D, A), (A, A, D))):
            F = sum(cart[x] * self.m[:, d, x][:, None] for x in range(3)) * -wJ[:, None]
            res = res + self._back(F, *o)
        mach2 = (rho * (vel * vel).sum(1) / (GAMMA * p)).max()
        return res, (wJ * rho, vel, p / rho, ek), mach2, ev.max()

    def _log_mean(self, a, b):
        f = (a - b) / (a + b)
        u = f * f
        series = 1.0 + u * (1.0 / 3.0 + u * (0.2 + u * (1.0 / 7.0 + u / 9.0)))
        safe = torch.where(u < 0.01, torch.full_like(f, 0.5), f)
        return 0.5 * (a + b) / torch.where(u < 0.01, series, torch.atanh(safe) / safe)

    def _faces(self, U, res):
        lift = [0.0]
        ev_max = torch.zeros((), dtype=torch.float64, device=self.dev)
        for d in range(3):
            axis = 2 - d
            left = lambda a: a.reshape(self.n + a.shape[1:]).roll(1, axis).reshape(a.shape)
            right = lambda a: a.reshape(self.n + a.shape[1:]).roll(-1, axis).reshape(a.shape)
            trace = []
            for s in (0, 1):        # min face of the element, max face of the one below it
                ops = [[self.A] * 3 for _ in range(4)]
                for a in range(4):
                    ops[a][d] = self.F[s:s + 1]
                    if a:
                        ops[a][a - 1] = self.dF[s:s + 1] if a - 1 == d else self.D
                t = [self._to(U, *o).reshape(self.E, 5, self.M, self.M) for o in ops]
                g = self._cartesian(t[1:], self.fm[d][s])
                trace.append([t[0]] + g if s == 0 else [left(x) for x in [t[0]] + g])
            VR, VL = trace[0][0], trace[1][0]
            G = [0.5 * (trace[0][1 + x] + trace[1][1 + x]) for x in range(3)]
            nn, area = left(self.fn[d][1]), left(self.fa[d][1])
            wA = self.w2 * area
            tau = (self.K ** 2) * self.flow.rel_penalty / torch.minimum(self.length[d], left(self.length[d]))
            les = 0.5 * (self.les + left(self.les))
            fl, sym, ev = self._flux(VL, VR, G, nn, wA, tau[:, None, None], les)
            ev_max = torch.maximum(ev_max, ev.max())
            for s in (0, 1):
                F, S = (fl, sym) if s == 0 else (right(fl), [right(x) for x in sym])
                c = self.fm[d][s].flatten(3)[:, :, :, :5]
                o = [self.A] * 3
                o[d] = self.F[s:s + 1]
                shape = [self.M] * 3
                shape[2 - d] = 1
                res = res + self._back((F * (1.0 if s else -1.0)).reshape([self.E, 5] + shape), *o)
                for a in range(3):
                    o = [self.A] * 3
                    o[d] = self.F[s:s + 1]
                    o[a] = self.dF[s:s + 1] if a == d else self.D
                    P = sum(S[x] * c[:, a, x][:, :, None, None] for x in range(3))
                    res = res + self._back(P.reshape([self.E, 5] + shape), *o)
        return res, ev_max

    def _flux(self, VL, VR, G, nn, wA, tau, les):
        rL, uL, pL, _ = self._primitive(VL)
        rR, uR, pR, _ = self._primitive(VR)
        dot = lambda a, b: (a * b).sum(1)
        z0 = ((rL / pL).sqrt(), (rR / pR).sqrt())
        z4 = ((rL * pL).sqrt(), (rR * pR).sqrt())
        z0A, z4A = 0.5 * (z0[0] + z0[1]), 0.5 * (z4[0] + z4[1])
        z0L, z4L = self._log_mean(*z0), self._log_mean(*z4)
        vel = 0.5 * (uL * z0[0][:, None] + uR * z0[1][:, None]) / z0A[:, None]
        rho, p1 = z0A * z4L, z4A / z0A
        p2 = 0.5 * ((GAMMA + 1.0) / GAMMA * z4L / z0L + 0.4 / GAMMA * p1)
        vn, kin = dot(vel, nn), 0.5 * dot(vel, vel)
        a2 = GAMMA * p2 / rho
        a, H = a2.sqrt(), a2 / 0.4 + kin
        E = H - p2 / rho
        dV = VR - VL
        m = rho * dot(vel, dV[:, 1:4])
        dr = m + rho * (dV[:, 0] + E * dV[:, 4])
        mom = vel * (m + rho * (dV[:, 0] + H * dV[:, 4]))[:, None] + p2[:, None] * dV[:, 1:4]
        dE = H * m + rho * E * (dV[:, 0] + H * dV[:, 4]) + p2 * kin * dV[:, 4]
        fac = 0.5 * (1.0 + 1.0 / 6.0)
        l1, l2, l3 = (vn + a).abs() * fac, (vn - a).abs() * fac, 0.5 * vn.abs()
        s, t = 0.5 * (l1 + l2), 0.5 * (l1 - l2)
        b4 = 0.4 * (kin * dr - dot(vel, mom) + dE)
        b5 = dot(nn, mom) - vn * dr
        b6 = (s - l3) * b4 / a2 + t * b5 / a
        b7 = t * b4 / a + (s - l3) * b5
        fl = [rho * vn - (l3 * dr + b6)]
        fl += [rho * vn * vel[:, i] + p1 * nn[:, i] - (l3 * mom[:, i] + vel[:, i] * b6 + nn[:, i] * b7) for i in range(3)]
        fl.append(rho * vn * H - (l3 * dE + H * b6 + vn * b7))
        # viscous flux on the averaged state
        Va = 0.5 * (VL + VR)
        rA, vel, _, _ = self._primitive(Va)
        ev = torch.zeros_like(rA)
        du, T, q = self._viscous(Va[:, 4], vel, G, self.mu, ev)
        if self.flow.sgs != "none":
            ev = self._eddy(rA, du, les)
            du, T, q = self._viscous(Va[:, 4], vel, G, self.mu, ev)
        for i in range(3):
            fl[1 + i] = fl[1 + i] - sum(T[i][x] * nn[:, x] for x in range(3))
        fl[4] = fl[4] - sum((sum(vel[:, i] * T[i][x] for i in range(3)) - q[x]) * nn[:, x] for x in range(3))
        fl = torch.stack(fl, 1) * wA[:, None]
        # penalty and symmetrising terms: the viscous tensor K of the averaged
        # state, K_xy dV = the viscous flux in x of a gradient dV along y
        muT = self.mu + ev
        kap = self.mu * GAMMA / 0.72 + ev * GAMMA / 0.9
        dV = VL - VR
        povr = -1.0 / Va[:, 4]

        def tensor(x, n):
            """Viscous flux in direction x of the gradient dV n, without muT p / rho."""
            g = [(dV[:, 1 + i] + vel[:, i] * dV[:, 4]) for i in range(3)]
            div = sum(g[i] * n[:, i] for i in range(3))
            t = [g[i] * n[:, x] + g[x] * n[:, i] + (-2.0 / 3.0 * div if i == x else 0.0) for i in range(3)]
            e = sum(vel[:, i] * t[i] for i in range(3)) + kap / muT * povr / 0.4 * dV[:, 4] * n[:, x]
            return torch.stack([torch.zeros_like(e)] + t + [e], 1)

        fact = (povr * wA * muT)[:, None]
        sym = [-0.5 * self.flow.theta_sym * fact * tensor(x, nn) for x in range(3)]
        # the penalty takes the normal-normal tensor with lambda + mu in the normal part
        g = [(dV[:, 1 + i] + vel[:, i] * dV[:, 4]) for i in range(3)]
        gn, un = sum(g[i] * nn[:, i] for i in range(3)), dot(vel, nn)
        pen = [torch.zeros_like(gn)] + [gn / 3.0 * nn[:, i] + g[i] for i in range(3)]
        pen.append(un / 3.0 * gn + sum(vel[:, i] * g[i] for i in range(3)) + kap / muT * povr / 0.4 * dV[:, 4])
        return fl + tau[:, None] * fact * torch.stack(pen, 1), sym, ev

    def _mass(self, prim, X):
        """Galerkin projection of w J dU/dV times the field of X."""
        r, vel, e, ek = prim                                   # w J rho, velocity, p / rho, kinetic energy
        V = self._to(X, self.A, self.A, self.A)
        E = e / 0.4 + ek
        uV = (vel * V[:, 1:4]).sum(1)
        y0 = r * (V[:, 0] + uV + E * V[:, 4])
        y = [y0] + [vel[:, i] * y0 + r * e * (V[:, 1 + i] + vel[:, i] * V[:, 4]) for i in range(3)]
        y.append(E * y0 + r * e * (uV + (E + ek) * V[:, 4]))
        return self._back(torch.stack(y, 1), self.A, self.A, self.A)

    def _solve(self, prim, b):
        """Conjugate gradients with the element means' dV/dU, to rounding."""
        wr, vel, e, ek = prim
        mean = lambda a: a.mean((-1, -2, -3))
        r, u, e0 = mean(wr / self.w3), mean(vel), mean(e)
        k, one = 0.5 * (u * u).sum(1), torch.ones_like(e0)
        H = torch.zeros(self.E, 5, 5, dtype=torch.float64, device=self.dev)
        Et = e0 / 0.4 + k
        col = torch.cat([one[:, None], u, Et[:, None]], 1)
        H += r[:, None, None] * col[:, :, None] * col[:, None, :]
        pr = (r * e0)[:, None]
        for i in range(3):
            H[:, 1 + i, 1 + i] += pr[:, 0]
            H[:, 1 + i, 4] += pr[:, 0] * u[:, i]
            H[:, 4, 1 + i] += pr[:, 0] * u[:, i]
        H[:, 4, 4] += pr[:, 0] * (Et + k)
        P = torch.linalg.inv(H.cpu()).to(self.dev)
        pre = lambda x: torch.matmul(P, x.flatten(2)).reshape(x.shape)
        dot = lambda a, c: (a * c).sum((1, 2, 3, 4), keepdim=True)
        x, res = torch.zeros_like(b), b
        z = pre(res)
        p, rz = z, dot(res, z)
        for _ in range(60):
            Ap = self._mass(prim, p)
            a = rz / dot(p, Ap).clamp_min(1e-300)
            x, res = x + a * p, res - a * Ap
            if bool((res.abs().amax() < 1e-14 * b.abs().amax())):
                break
            z = pre(res)
            new = dot(res, z)
            p, rz = z + new / rz.clamp_min(1e-300) * p, new
        return x

    def residual(self, U):
        res, prim, mach2, ev = self._volume(U)
        res, evf = self._faces(U, res)
        return self._solve(prim, res), mach2, torch.maximum(ev, evf)

    def steps(self, U, count):
        R, mach2, ev = self.residual(U)
        for _ in range(count):
            U0 = U
            for a, b in RK:
                U = (1.0 - a) * U + a * U0 - b * self.dt * R
                R, mach2, ev = self.residual(U)
        return U, mach2, ev


def exact(case, seed):
    """What run returns, for the periodic cases of up to 9,000 elements: the
    headline size takes a minute in dense tensor algebra, and the open box
    carries its characteristic boundary states and sponge besides."""
    if case["flow"] == "box":
        return None
    flows = _flows(case, seed)
    if sum(f.n_elems * f.n_dofs for f in flows) * max(1, case.get("steps", 0)) > 3.1e7:
        return None
    out = []
    for flow in flows:
        ref = _Plain(flow)
        U = ref.start()
        if case["mode"] == "residual":
            R, mach2, ev = ref.residual(U)
        else:
            R, mach2, ev = ref.steps(U, case["steps"])
        monitoring = torch.zeros(8, dtype=torch.float64)
        monitoring[6] = mach2.cpu()
        if case.get("sgs", "none") != "none":
            monitoring[7] = ev.cpu()
        out.append((R.reshape(flow.n_elems, 5, flow.n_dofs).cpu(), monitoring))
    if case["mode"] == "residual":
        return dict(residual=out[0][0], monitoring=out[0][1])
    if case["mode"] == "batch":
        return dict(solution=[u for u, _ in out])
    return dict(solution=out[0][0], monitoring=out[0][1], rk_steps=None)
