"""The work that a user of sod2d_amd has it do, as cases for timing.

Four kinds, each through the public Python entry points:

  step     one time step of a periodic Taylor-Green run (solver.TGVRun.step):
           the Runge-Kutta stages with the fused right-hand side, the entropy
           residual, the entropy-viscosity sensor and, where "adaptive", the
           CFL time step read back to the host.  The plain path (FP64 or FP32
           operators) and the LPS-stabilised path with the live sensor.
  rhs      the drop-in operators as a host's updateF calls them: convection,
           viscous operator added to it, lumped solve with the stage update.
  stab     the drop-in LPS operators: time scale, projections, stabilised
           viscous operator.
  monitor  what a run prints between steps: kinetic energy, dissipation rate,
           largest Mach number, and the CFL time step.

Sizes: elements per direction of a structured box and the order p (2, 3, 4, all
that the kernels take; 4 is the default order, 3 the benchmark's).
"""
import math

import numpy as np
import torch

from sod2d_amd import case as case_mod
from sod2d_amd import device as dev
from sod2d_amd import solver

F64 = torch.float64
TWO_PI = 2.0 * math.pi


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: a debugging or regression box, bound by latency,
        # launches and the read-back of the time step
        dict(name="step_p3_tiny", kind="step", p=3, nx=8, ny=8, nz=8, precision=8, lps=False,
             parity=False, adaptive=True, mach=0.3),
        # the headline benchmark: 64^3 elements, p = 3, FP64, fixed time step
        dict(name="step_p3_64", kind="step", p=3, nx=64, ny=64, nz=64, precision=8, lps=False,
             parity=True, adaptive=False, mach=0.1),
        # the FP32-operator mode on a ragged box, adaptive time step
        dict(name="step_p3_fp32op", kind="step", p=3, nx=45, ny=38, nz=51, precision=4, lps=False,
             parity=False, adaptive=True, mach=0.2),
        # the compressible regression case: 12^3 elements, p = 4, LPS, M = 1.25
        dict(name="step_p4_lps_12", kind="step", p=4, nx=12, ny=12, nz=12, precision=8, lps=True,
             parity=True, adaptive=True, mach=1.25),
        # a production-size run of the default (LPS, live sensor) path at p = 4
        dict(name="step_p4_lps_35", kind="step", p=4, nx=35, ny=31, nz=38, precision=8, lps=True,
             parity=True, adaptive=True, mach=0.4),
        # the LPS path at p = 3, fixed time step (the benchmark's LPS mode)
        dict(name="step_p3_lps_48", kind="step", p=3, nx=48, ny=48, nz=48, precision=8, lps=True,
             parity=True, adaptive=False, mach=0.1),
        # the plain path at the other orders, ragged boxes
        dict(name="step_p4_plain", kind="step", p=4, nx=33, ny=40, nz=36, precision=8, lps=False,
             parity=False, adaptive=True, mach=0.2),
        dict(name="step_p2_plain", kind="step", p=2, nx=53, ny=61, nz=47, precision=8, lps=False,
             parity=False, adaptive=True, mach=0.2),
        # drop-in operators on distorted elements, mu_sgs present; the largest
        dict(name="rhs_p3_f64", kind="rhs", p=3, nx=80, ny=96, nz=72, dtype="float64", sgs=True),
        dict(name="rhs_p4_f64", kind="rhs", p=4, nx=40, ny=44, nz=36, dtype="float64", sgs=False),
        # a single-precision host (the default real(4) build), default order
        dict(name="rhs_p4_f32", kind="rhs", p=4, nx=37, ny=29, nz=43, dtype="float32", sgs=True),
        # drop-in LPS operators at the default order
        dict(name="stab_p4_f64", kind="stab", p=4, nx=30, ny=27, nz=34, sgs=False),
    ]


def _box(rng, p, lo, hi):
    """Elements per direction, near a number of element-nodes spread over lo..hi
    in the logarithm, with different counts per direction."""
    en = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    m = (en / (p + 1) ** 3) ** (1.0 / 3.0)
    return [max(3, round(m * rng.uniform(0.8, 1.2))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["step", "step", "step", "rhs", "rhs", "stab", "monitor"])
    p = rng.choice([2, 3, 3, 4, 4])
    if kind == "step":
        lps = rng.random() < 0.4
        n = _box(rng, p, 30e3, 4e6 if lps else 9e6)
        return dict(kind=kind, p=p, nx=n[0], ny=n[1], nz=n[2],
                    precision=8 if lps else rng.choice([8, 8, 4]), lps=lps,
                    parity=rng.random() < 0.5, adaptive=rng.random() < 0.5,
                    mach=round(rng.uniform(0.1, 1.25), 3))
    n = _box(rng, p, 30e3, 15e6 if kind == "rhs" else 6e6)
    c = dict(kind=kind, p=p, nx=n[0], ny=n[1], nz=n[2])
    if kind == "rhs":
        c["dtype"] = rng.choice(["float64", "float64", "float32"])
    if kind == "monitor":
        c["mach"] = round(rng.uniform(0.1, 1.25), 3)
    else:
        c["sgs"] = rng.random() < 0.5
    return c


# ------------------------------------------------------------------ inputs
_geometry = {}  # the last mesh on the host: a run keeps its mesh from step to step


def _geo(case):
    """Periodic box for the runs; distorted, non-periodic box for the operators."""
    run = case["kind"] in ("step", "monitor")
    key = (case["p"], case["nx"], case["ny"], case["nz"], run)
    if key not in _geometry:
        _geometry.clear()
        _geometry[key] = case_mod.build_case(
            case["p"], (case["nx"], case["ny"], case["nz"]), periodic=run, lengths=(TWO_PI,) * 3,
            jitter=0.0 if run else (0.05 if case["p"] < 4 else 0.03), seed=2)
    return _geometry[key]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _initial(coord, t, seed):
    """A Taylor-Green vortex with a few random solenoidal modes and entropy
    and pressure fluctuations on it (the state of a run under way), on the GPU."""
    r = np.random.default_rng(seed)
    x = torch.from_numpy(np.ascontiguousarray(coord.T)).cuda()
    n = x.shape[1]
    u = torch.zeros(3, n, dtype=F64, device="cuda")
    u[0] = torch.sin(x[0]) * torch.cos(x[1]) * torch.cos(x[2])
    u[1] = -torch.cos(x[0]) * torch.sin(x[1]) * torch.cos(x[2])
    p = (torch.cos(2 * x[0]) + torch.cos(2 * x[1])) * (torch.cos(2 * x[2]) + 2.0) / 16.0
    s = torch.zeros(n, dtype=F64, device="cuda")
    for _ in range(5):
        k = r.integers(-4, 5, 3).astype(float)
        k[int(r.integers(0, 3))] = float(r.integers(1, 5))
        a = np.cross(k, r.normal(size=3))
        a *= 0.15 / np.linalg.norm(a)
        c = torch.cos(k[0] * x[0] + k[1] * x[1] + k[2] * x[2] + r.uniform(0, TWO_PI))
        for d in range(3):
            u[d] += float(a[d]) * c
        p += 0.02 * float(r.uniform(-1, 1)) * c
        s += 0.02 * float(r.uniform(-1, 1)) * c
    g = t.gamma_gas
    pr = t.po * torch.exp(p / t.po)
    rho = t.rho0 * (pr / t.po) ** (1.0 / g) * torch.exp(-s)
    uu = (u * u).sum(0)
    e_int = pr / (rho * (g - 1.0))
    cs = torch.sqrt(g * pr / rho)
    out = dict(u=u, q=rho * u, rho=rho, pr=pr, E=rho * (0.5 * uu + e_int), e_int=e_int,
               Tem=pr / (rho * t.Rgas), csound=cs, machno=torch.sqrt(uu) / cs,
               eta=rho / (g - 1.0) * torch.log(pr / t.po / (rho / t.rho0) ** g))
    return {k: v.cpu().numpy().T for k, v in out.items()}  # (npoin[,3]), Fortran order


def _params(case):
    return solver.TGVParams(M=case["mach"])


def _run(case, seed):
    geo, t = _geo(case), _params(case)
    more = dict(lps=True, sensor_path="live", high_mach=case["mach"] > 1.0) if case.get("lps") else {}
    return solver.TGVRun(
        case["p"], geometry=geo, params=t, initial=_initial(geo.mesh.coord, t, seed),
        op_precision=case.get("precision", 8), parity=case.get("parity", True),
        dt_mode="adaptive" if case.get("adaptive") else "fixed", **more)


def _sensor_field(n, seed):
    return 1e-3 * torch.rand(n, generator=_gen(seed), dtype=F64, device="cuda")


GAS = dict(gamma=1.4, Rgas=1.0, Cp=3.5, Pr=0.71)


def _operator_inputs(case, seed):
    """Random fields as the operator benchmark draws them, on the GPU, flat in the
    Fortran order of the reference's arrays."""
    geo, g = _geo(case), _gen(seed)
    m, T = geo.mesh, geo.tables
    n, ne, nn = m.npoin, m.nelem, T.nnode
    dt = torch.float32 if case.get("dtype") == "float32" else F64

    def uni(k, lo, hi):
        return (torch.rand(k, generator=g, dtype=F64, device="cuda") * (hi - lo) + lo).to(dt)

    a = dict(rho=uni(n, 0.9, 1.1),
             u=(0.3 * torch.randn(3 * n, generator=g, dtype=F64, device="cuda")).to(dt),
             pr=uni(n, 0.9 / 1.4, 1.1 / 1.4), mu_fluid=uni(n, 1e-4, 2e-4),
             mu_e=uni(ne * nn, 0.0, 1e-3),
             mu_sgs=uni(ne * nn, 0.0, 1e-4) if case["sgs"] else None)
    a["q"] = (a["rho"] * a["u"].view(3, n)).view(-1)
    a["h"] = 3.5 * a["pr"] / a["rho"]
    a["Tem"] = a["pr"] / a["rho"]
    a["E"] = a["pr"] / 0.4 + 0.5 * a["rho"] * (a["u"].view(3, n) ** 2).sum(0)
    up = dev.to_dev
    a.update(connec=up(m.connec), lpoin_w=up(m.lpoin_w), He=up(geo.He).to(dt),
             gpvol=up(geo.gpvol).to(dt), dl=up(T.dlxigp_ip).to(dt), invMl=up(geo.invMl).to(dt),
             helem=up(geo.helem).to(dt),
             tabs=[up(x) for x in (T.invAtoIJK, T.gmshAtoI, T.gmshAtoJ, T.gmshAtoK)])
    return geo, dt, a


def prepare(case, seed):
    if case["kind"] in ("step", "monitor"):
        run = _run(case, seed)
        if case["kind"] == "monitor":
            # an entropy viscosity, as the sensor leaves it
            run.mu_e.copy_(_sensor_field(run.mu_e.numel(), seed))
        return dict(case=case, run=run)
    geo, dt, a = _operator_inputs(case, seed)
    n = geo.mesh.npoin

    def z(k):
        return torch.zeros(k, dtype=dt, device="cuda")

    a.update(Rmass=z(n), Rmom=z(3 * n), Rener=z(n), case=case, nelem=geo.mesh.nelem, npoin=n,
             npoin_w=geo.mesh.npoin_w)
    if case["kind"] == "rhs":
        a.update(y=[a["rho"].clone(), a["q"].clone(), a["E"].clone()])
    else:
        a.update(tau=z(geo.mesh.nelem), proj=[z(3 * n) for _ in range(5)],
                 csound=torch.sqrt(1.4 * a["pr"] / a["rho"]))
    return a


# ------------------------------------------------------------------ one pass
DT, GAM = 1e-3, 0.3


def run(s):
    case = s["case"]
    if case["kind"] == "step":
        r = s["run"]
        r.step()
        return dict(rho=r.rho[1], q=r.q[1], E=r.E[1], mu_e=r.mu_e, dt=r.dt)
    if case["kind"] == "monitor":
        r = s["run"]
        return dict(r.diagnostics(), dt=r.adapt_dt())
    geo = (s["nelem"], s["npoin"], s["connec"])
    tabs = (s["dl"], *s["tabs"])
    R = (s["Rmass"], s["Rmom"], s["Rener"])
    if case["kind"] == "rhs":
        dev.full_convec_ijk(*geo, None, None, s["He"], s["gpvol"], s["dl"], None, *s["tabs"],
                            s["u"], s["q"], s["rho"], s["pr"], s["h"], *R, initialze=True,
                            fact=-1.0)
        dev.full_diffusion_ijk(*geo, None, s["He"], s["gpvol"], *tabs, GAS["Cp"], GAS["Pr"],
                               s["rho"], s["rho"], s["u"], s["Tem"], s["mu_fluid"], s["mu_e"],
                               s["mu_sgs"], None, *R, initialze=False, fact=-1.0)
        if case["dtype"] == "float32":
            return R  # the node updates take FP64 arrays
        dev.rk_stage_update(s["npoin"], s["npoin_w"], s["lpoin_w"], s["invMl"], DT, 1.0, 0.0, GAM,
                            s["rho"], s["q"], s["E"], *s["y"], *R)
        return (*R, *s["y"])
    dev.comp_tau(*geo, s["csound"], s["u"], s["helem"], 0.0, s["tau"])
    dev.full_proj_ijk(s["nelem"], s["npoin"], s["npoin_w"], s["connec"], s["lpoin_w"], None,
                      s["He"], s["gpvol"], *tabs, GAS["Cp"], GAS["Pr"], s["rho"], s["u"],
                      s["Tem"], None, s["invMl"], *s["proj"])
    dev.full_diff_stab_ijk(*geo, None, s["He"], s["gpvol"], *tabs, GAS["Cp"], GAS["Pr"],
                           s["rho"], s["rho"], s["u"], s["Tem"], s["mu_fluid"], s["mu_e"],
                           s["mu_sgs"], None, *s["proj"], s["tau"], *R, initialze=True, fact=-1.0)
    return (s["tau"], *s["proj"], *R)


# ------------------------------------------------------------------ least work
def _counts(case):
    p = case["p"]
    ne = case["nx"] * case["ny"] * case["nz"]
    n = ne * p ** 3
    if case["kind"] in ("rhs", "stab"):
        n = (case["nx"] * p + 1) * (case["ny"] * p + 1) * (case["nz"] * p + 1)
    return p, ne, ne * (p + 1) ** 3, n


def work(case):
    p, ne, en, n = _counts(case)
    # multiply-adds per element-node: convection, viscous operator, gradients of
    # the projections; per line 3 (p+1) neighbours (own node included)
    l = 3 * (p + 1)
    conv, diff, grad = 22 * l + 60, 11 * l + 130, 5 * l + 60
    if case["kind"] == "step":
        s = case["precision"]
        # per RHS: He, gpvol, mu_e, connectivity once per element-node; the state,
        # the base state and the new state, and the inverse mass per node
        rhs = (11 * s + 4) * en + 16 * 8 * n
        frhs = en * (conv + diff + (grad if case["lps"] else 0))
        # entropy residual (geometry again) and sensor
        rest = (80 + 4) * en + 12 * 8 * n + (8 + 8 + (0 if case["lps"] else 8)) * en + 8 * 8 * n
        stages = 4 if case["parity"] else 5
        return dict(bytes=stages * rhs + rest, flops=2.0 * (stages * frhs + en * (7 * l + 60)))
    if case["kind"] == "monitor":
        return dict(bytes=(80 + 8 + 4) * en + 8 * 8 * n, flops=2.0 * en * (3 * l + 60))
    if case["kind"] == "rhs":
        s = 4 if case["dtype"] == "float32" else 8
        geom = 10 * s * en + 4 * en + (s if case["sgs"] else 0) * en + s * en
        return dict(bytes=geom + (10 + 5 + (16 if s == 8 else 0)) * s * n,
                    flops=2.0 * en * (conv + diff))
    geom = (80 + 4 + 8 + (8 if case["sgs"] else 0)) * en
    return dict(bytes=geom + (8 + 15 + 5) * 8 * n, flops=2.0 * en * (diff + 2 * grad))


# ------------------------------------------------------------------ in plain torch
class _Plain:
    """The operators written out in torch, FP64, from their definitions: nodal
    fields gathered to (element, K, J, I) arrays, one-dimensional derivative
    matrices along each axis, sums back to the nodes."""

    def __init__(self, geo):
        m, T = geo.mesh, geo.tables
        self.p, n1 = geo.tables.porder, geo.tables.porder + 1
        self.n1, self.nn, self.ne, self.npoin = n1, n1 ** 3, m.nelem, m.npoin
        lex = np.argsort((T.gmshAtoI - 1) + n1 * ((T.gmshAtoJ - 1) + n1 * (T.gmshAtoK - 1)))
        self.lex = torch.from_numpy(lex.astype(np.int64)).cuda()
        con = torch.from_numpy(np.ascontiguousarray(m.connec.T)).cuda().long() - 1
        self.con = con.T[:, self.lex].contiguous().view(self.ne, n1, n1, n1)
        self.w = torch.from_numpy(m.lpoin_w.astype(np.int64)).cuda() - 1
        He = torch.from_numpy(geo.He.ravel(order="F")).cuda().view(self.ne, self.nn, 3, 3)
        self.He = He[:, self.lex].contiguous().view(self.ne, n1, n1, n1, 3, 3)  # [..., j, i]
        vol = torch.from_numpy(geo.gpvol.ravel(order="F")).cuda().view(self.ne, self.nn)
        self.vol = vol[:, self.lex].contiguous().view(self.ne, n1, n1, n1)
        D = np.zeros((n1, n1))
        for a in range(self.nn):
            D[T.gmshAtoI[a] - 1] = T.dlxigp_ip[a, 0]
        self.D = torch.from_numpy(D).cuda()
        self.invMl = torch.from_numpy(geo.invMl).cuda()
        self.h = torch.from_numpy(geo.helem).cuda()

    def e(self, f):
        return f[self.con]

    def el(self, a):
        """(nelem, nnode) column-major element array -> (element, K, J, I)."""
        return a.double().view(self.nn, self.ne).T[:, self.lex].view(self.con.shape)

    def un(self, a):
        """The inverse of el, flat."""
        out = torch.empty(self.nn, self.ne, dtype=F64, device="cuda")
        out[self.lex] = a.reshape(self.ne, self.nn).T.contiguous()
        return out.view(-1)

    def lines(self, f, D):
        """D along I, J and K."""
        n1, ne = self.n1, self.ne
        return ((f.reshape(-1, n1) @ D.T.contiguous()).view_as(f),
                torch.matmul(D, f.reshape(-1, n1, n1)).view_as(f),
                torch.matmul(D, f.reshape(ne, n1, n1 * n1)).view_as(f))

    def grad(self, f):
        d = self.lines(f, self.D)
        return [sum(self.He[..., j, i] * d[j] for j in range(3)) for i in range(3)]

    def div(self, F):
        return sum(self.grad(F[i])[i] for i in range(3))

    def weak(self, F):
        """sum_k sum_b dl(b,k,.) gpvol sum_d He(d,k) F_d at b."""
        out = 0.0
        for k in range(3):
            G = self.vol * sum(self.He[..., k, d] * F[d] for d in range(3))
            out = out + self.lines(G, self.D.T.contiguous())[k]
        return out

    def add(self, r):
        return torch.zeros(self.npoin, dtype=F64, device="cuda").index_add_(
            0, self.con.reshape(-1), r.reshape(-1))

    def convec(self, rho, u, q, pr, h):
        """full_convec_ijk: mass, momentum, energy (element values, times gpvol)."""
        E = self.e
        r, p = E(rho), E(pr)
        U, Q = [E(u[d]) for d in range(3)], [E(q[d]) for d in range(3)]
        H = E(h) + 0.5 * sum(x * x for x in U)
        rH = r * H
        dot = lambda a, g: sum(a[j] * g[j] for j in range(3))  # noqa: E731
        gr, gp, gH, grH = (self.grad(x) for x in (r, p, H, rH))
        gU, gQ = [self.grad(x) for x in U], [self.grad(x) for x in Q]
        dU, dQ = sum(gU[i][i] for i in range(3)), sum(gQ[i][i] for i in range(3))
        ur = dot(U, gr)
        mass = 0.5 * (dQ + r * dU + ur)
        mom = [0.25 * (self.div([Q[i] * v for v in U]) + U[i] * dQ + Q[i] * dU +
                       r * self.div([U[i] * v for v in U]) + U[i] * ur + dot(Q, gU[i]) +
                       dot(U, gQ[i])) + gp[i] for i in range(3)]
        ener = 0.25 * (self.div([rH * v for v in U]) + H * dQ + rH * dU +
                       r * self.div([H * v for v in U]) + dot(Q, gH) + dot(U, grH) + H * ur)
        return [self.vol * x for x in (mass, *mom, ener)]

    def strain(self, gU):
        dv = sum(gU[i][i] for i in range(3))
        return dv, [[gU[i][j] + gU[j][i] for j in range(3)] for i in range(3)]

    def diffu(self, rho, u, Tem, muf, mue, sgs, Cp, Pr):
        """full_diffusion_ijk (element values)."""
        E = self.e
        r, mf, U = E(rho), E(muf), [E(u[d]) for d in range(3)]
        dv, S = self.strain([self.grad(x) for x in U])
        mg = mf + r * sgs
        tau = [[(mg + mue) * S[i][j] - (mg * (2.0 / 3.0) * dv if i == j else 0.0)
                for j in range(3)] for i in range(3)]
        tu = [sum(tau[i][j] * U[j] for j in range(3)) for i in range(3)]
        kappa = mf * Cp / Pr + mue * Cp / Pr + Cp * r * sgs / 0.9
        return [mue / r * self.weak(self.grad(r)), *[self.weak(tau[i]) for i in range(3)],
                self.weak(tu) + kappa * self.weak(self.grad(E(Tem)))]

    def lumped(self, f):
        out = f.clone()
        out[self.w] = f[self.w] * self.invMl[self.w]
        return out

    def proj(self, rho, u, Tem):
        """full_proj_ijk: ProjMass, ProjEner, ProjMX, MY, MZ, each [3] of nodal fields."""
        E = self.e
        dv, S = self.strain([self.grad(E(u[d])) for d in range(3)])
        t = [[S[i][j] - ((2.0 / 3.0) * dv if i == j else 0.0) for j in range(3)] for i in range(3)]
        return [[self.lumped(self.add(self.vol * x)) for x in g]
                for g in (self.grad(E(rho)), self.grad(E(Tem)), *t)]

    def tau(self, cs, u, c=0.5):
        sp = cs + torch.sqrt((u * u).sum(0))
        return self.h * (c / self.p) * self.e(sp).reshape(self.ne, -1).amax(1)

    def stab(self, rho, u, Tem, muf, mue, sgs, proj, tau, Cp, Pr, c_lps=float(np.float32(0.1))):
        """full_diff_stab_ijk (element values)."""
        E = self.e
        r, mf, U = E(rho), E(muf), [E(u[d]) for d in range(3)]
        gr, gT = self.grad(r), self.grad(E(Tem))
        dv, S = self.strain([self.grad(x) for x in U])
        mg = mf + r * sgs
        cl = (-c_lps * tau).view(-1, 1, 1, 1)
        kappa = mf * Cp / Pr + mue * Cp / Pr + Cp * r * sgs / 0.9
        tw = [[(mg + mue) * S[i][j] - (mg * (2.0 / 3.0) * dv if i == j else 0.0)
               for j in range(3)] for i in range(3)]
        M = [[cl * (E(proj[2 + i][d]) - (S[i][d] - ((2.0 / 3.0) * dv if i == d else 0.0))) * r +
              tw[i][d] for d in range(3)] for i in range(3)]
        F0 = [cl * (E(proj[0][d]) - gr[d]) + mue / r * gr[d] for d in range(3)]
        F4 = [cl * (E(proj[1][d]) - gT[d]) * r * Cp / Pr + kappa * gT[d] +
              sum(tw[d][j] * U[j] for j in range(3)) for d in range(3)]
        return [self.weak(F0), *[self.weak(M[i]) for i in range(3)], self.weak(F4)]

    def scalar(self, eta, u):
        """The lumped convective residual of the entropy with the flux u*eta."""
        E = self.e
        U, s = [E(u[d]) for d in range(3)], E(eta)
        gs = self.grad(s)
        r = 0.5 * (self.div([v * s for v in U]) + s * sum(self.grad(U[i])[i] for i in range(3)) +
                   sum(U[i] * gs[i] for i in range(3)))
        return self.lumped(self.add(self.vol * r))

    def per_elem(self, x):
        return x.view(-1, 1, 1, 1)

    def norm(self, eta):
        v = eta[self.w]
        return (v - v.mean()).abs().max()


class _PlainRun:
    """The first time step of a run, in plain torch."""

    A = [0.0, 0.443568244942995, 0.291111420073766, 0.270612601278217, 0.110577759392786,
         0.458557505351052]  # gamma_{s,s-1} of the SSP(5,3) scheme

    def __init__(self, case, seed):
        self.case, geo = case, _geo(case)
        self.P = P = _Plain(geo)
        mach, g = case["mach"], 1.4
        Cp, self.Pr, self.g = 1004.0, 0.71, g
        self.Cp, self.R = Cp, Cp * (g - 1.0) / g
        T0 = 1.0 / (g * self.R * mach * mach)
        self.po = self.R * T0
        self.mf = (1.0 / 1600.0) / (0.000001458 * T0 ** 1.5 / (T0 + 110.40))
        ic = _initial(geo.mesh.coord, _params(case), seed)
        up = lambda k: torch.from_numpy(np.ascontiguousarray(ic[k].T)).cuda()  # noqa: E731
        self.ic = {k: up(k) for k in ic}
        self.helem_l = P.el(torch.from_numpy(geo.helem_l.ravel(order="F")).cuda())
        self.lps = case.get("lps", False)
        if self.lps:
            self.Ml = torch.from_numpy(geo.Ml).cuda()
            self.count = P.add(torch.ones_like(P.vol))
        self.high = mach > 1.0
        self.ce = 0.1

    def suth(self, T):
        return self.mf * 0.000001458 * T ** 1.5 / (T + 110.4)

    def eos(self, y, old):
        """u, p, T, c at the working nodes; old values elsewhere."""
        w = self.P.w
        u, p, T, c = (x.clone() for x in old)
        r, q, E = y[0][w], y[1:4][:, w], y[4][w]
        v = q / r
        e = E / r - 0.5 * (v * v).sum(0)
        u[:, w] = v
        p[w] = r * (self.g - 1.0) * e
        T[w] = (self.g - 1.0) * e / self.R
        c[w] = torch.sqrt(self.g * (self.g - 1.0) * e)
        return u, p, T, c

    def dt(self, u, cs, T, mu, rho):
        P = self.P
        hh = P.h / (2.0 * P.p + 1.0)
        L3 = (u.abs().amax(0) + cs)[P.con].reshape(P.ne, -1).amax(1)
        a = (0.5 * hh / L3).min()
        mx = ((P.e(self.suth(T)) + mu) / P.e(rho)).reshape(P.ne, -1).amax(1)
        return torch.minimum(a, (0.5 * hh * hh / mx).min()).item()

    def sensor(self, Reta, rho, u, T, cs, eta, live_end=False):
        P, p = self.P, self.P.p
        hk = P.per_elem(P.h)
        if self.lps:
            if self.high:
                norm, self.ce = rho[P.w].min(), 1.0
            else:
                norm = P.norm(eta)
            speed = torch.sqrt((u * u).sum(0)) + cs
        else:
            norm = P.norm(eta)
            speed = torch.sqrt((u * u).sum(0)) + torch.sqrt(self.R * self.g * T)
        beta = P.per_elem((P.e(rho * speed) * hk * (0.5 / p)).reshape(P.ne, -1).amax(1))
        h = hk / p if self.lps else self.helem_l
        mu = torch.minimum(self.ce * P.e(rho * Reta.abs() / norm) * h * h, beta)
        if not self.lps:
            return self.filter(mu)
        if not live_end:
            return mu
        gU = [P.grad(P.e(u[d])) for d in range(3)]
        dv = P.add(P.vol * sum(gU[i][i] for i in range(3))) / self.Ml
        cw = [gU[1][2] - gU[2][1], gU[2][0] - gU[0][2], gU[0][1] - gU[1][0]]
        om = sum((P.add(c) / self.count) ** 2 for c in cw)
        eps = float(np.finfo(np.float64).eps)
        d2 = dv * dv
        phi = torch.clamp((4.0 / 3.0) * d2 / (d2 + om + eps), max=1.0)
        t = P.e(torch.sqrt((u * u).sum(0))) / self.helem_l
        phi2 = P.e(d2) / (P.e(d2) + t * t + eps)
        return mu * (torch.clamp(P.e(phi) - 0.1, min=0.0) * phi2 + 0.1)

    def filter(self, mu):
        """The 3x3x3 filter (1/4, 1/2, 1/4 per direction) over the geometric order of
        the line positions (first, inner ones, last); beyond the ends the reference
        reads its line indices 3 and p (from 1)."""
        n1 = self.P.n1
        pos = [0, *range(2, n1), 1]  # line index at each geometric position
        F = torch.zeros(n1, n1, dtype=F64, device="cuda")
        for g in range(n1):
            for o, wt in ((-1, 0.25), (0, 0.5), (1, 0.25)):
                s = g + o
                F[pos[g], 2 if s < 0 else (n1 - 2 if s >= n1 else pos[s])] += wt
        for axis in range(3):
            mu = self.P.lines(mu, F)[axis]
        return mu

    def first(self):
        ic = self.ic
        return torch.stack([ic["rho"], *ic["q"], ic["E"]]), (ic["u"], ic["pr"], ic["Tem"],
                                                               ic["csound"])

    def step(self):
        P, ic = self.P, self.ic
        y0, prim0 = self.first()
        u0, _, T0, c0 = prim0
        rho0, eta0 = ic["rho"], ic["eta"]
        dt = self.dt(u0, c0, T0, torch.zeros_like(P.vol), rho0)
        tau = P.tau(c0, u0) if self.lps else None
        R1 = P.scalar(eta0, u0)
        mu = self.sensor(R1, rho0, u0, T0, c0, eta0)

        def rhs(y):
            u, p, T, _ = self.eos(y, prim0)
            rho, q, muf = y[0], y[1:4], self.suth(T)
            h = self.g / (self.g - 1.0) * p / rho
            C = P.convec(rho, u, q, p, h)
            if self.lps:
                V = P.stab(rho, u, T, muf, mu, 0.0, P.proj(rho, u, T), tau, self.Cp, self.Pr)
            else:
                V = P.diffu(rho, u, T, muf, mu, 0.0, self.Cp, self.Pr)
            return torch.stack([-P.lumped(P.add(c + v)) for c, v in zip(C, V)])

        def comb(l1, ls, gam, y, R):
            out, w = y.clone(), P.w
            out[:, w] = l1 * y0[:, w] + ls * y[:, w] + gam * dt * R[:, w]
            return out

        y = comb(1.0, 0.0, self.A[1], y0, rhs(y0))
        for s in range(2, 6):
            l1, ls = (0.571403511494104, 0.428596488505896) if s == 4 else (0.0, 1.0)
            y = comb(l1, ls, self.A[s], y, rhs(y))
        u, p, T, cs = self.eos(y, prim0)
        eta = eta0.clone()
        w = P.w
        eta[w] = y[0][w] / (self.g - 1.0) * torch.log(p[w] / self.po / y[0][w] ** self.g)
        R2 = P.scalar(eta0, u0)
        aux = torch.zeros_like(eta)
        aux[w] = 1.5 * R2[w] - 0.5 * R1[w] + (eta[w] - eta0[w]) / dt
        mu = self.sensor(aux, y[0], u, T, cs, eta, live_end=True)
        if self.case["adaptive"]:
            dt = self.dt(u, cs, T, mu, y[0])
        return dict(rho=y[0], q=y[1:4].reshape(-1), E=y[4], mu_e=P.un(mu), dt=dt)

    def monitor(self, mu):
        P, ic = self.P, self.ic
        u, rho = ic["u"], ic["rho"]
        gU = [P.grad(P.e(u[d])) for d in range(3)]
        mf = P.e(self.suth(ic["Tem"]))
        dv = sum(gU[i][i] for i in range(3))
        w2 = ((gU[2][1] - gU[1][2]) ** 2 + (gU[0][2] - gU[2][0]) ** 2 +
              (gU[1][0] - gU[0][1]) ** 2)
        # the case's own roundings of pi and of 4/3 (a single-precision constant)
        S = ((P.vol * (mf + mu) * w2).sum() / P.vol.sum()).item()
        Dl = float(np.float32(4.0 / 3.0)) * ((P.vol * mf * dv * dv).sum() / P.vol.sum()).item()
        ek = (P.vol * P.e(0.5 * rho * (u * u).sum(0))).sum().item() / (2.0 * 3.14159) ** 3
        return dict(time=0.0, EK=ek, eps_S=S, eps_D=Dl, eps_T=S + Dl,
                    maxmach=ic["machno"][P.w].max().item(),
                    dt=self.dt(u, ic["csound"], ic["Tem"], mu, rho))


def exact(case, seed):
    if case["kind"] == "step":
        return _PlainRun(case, seed).step()
    if case["kind"] == "monitor":
        plain = _PlainRun(case, seed)
        return plain.monitor(plain.P.el(_sensor_field(plain.P.ne * plain.P.nn, seed)))
    geo, _, a = _operator_inputs(case, seed)
    P = _Plain(geo)
    n = P.npoin
    d = {k: a[k].double() for k in ("rho", "u", "pr", "mu_fluid", "q", "h", "Tem", "E")}
    u, q = d["u"].view(3, n), d["q"].view(3, n)
    sgs = P.el(a["mu_sgs"]) if case["sgs"] else 0.0
    mue = P.el(a["mu_e"])
    if case["kind"] == "rhs":
        if case["dtype"] == "float32":  # the geometry as the call receives it
            P.He, P.vol, P.D = (x.float().double() for x in (P.He, P.vol, P.D))
        C = P.convec(d["rho"], u, q, d["pr"], d["h"])
        V = P.diffu(d["rho"], u, d["Tem"], d["mu_fluid"], mue, sgs, GAS["Cp"], GAS["Pr"])
        R = [-P.add(c + v) for c, v in zip(C, V)]
        if case["dtype"] == "float32":
            return R[0], torch.cat(R[1:4]), R[4]
        R = [P.lumped(r) for r in R]
        y = [b + GAM * DT * r for b, r in zip((d["rho"], *q, d["E"]), R)]
        return R[0], torch.cat(R[1:4]), R[4], y[0], torch.cat(y[1:4]), y[4]
    tau = P.tau(torch.sqrt(1.4 * d["pr"] / d["rho"]), u)
    proj = P.proj(d["rho"], u, d["Tem"])
    V = P.stab(d["rho"], u, d["Tem"], d["mu_fluid"], mue, sgs, proj, tau, GAS["Cp"], GAS["Pr"])
    R = [-P.add(v) for v in V]
    return (tau, *[torch.cat(x) for x in proj], R[0], torch.cat(R[1:4]), R[4])
