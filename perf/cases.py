"""The work that programs built on this framework have it do, for timing.

A program holds the static inputs of a grid (numbering, metric, mass, layer
sizes), a state and the work arrays, creates a context for them, and then
steps the state (``TimeStepper``, ``RosenbrockSchur``, a replayed step graph
of an ensemble), calls the drop-in parts of the step from an integrator of
its own (``FcnPrepareGPU`` + ``FcnGPU``, ``JacSchurGPU`` + ``SchurSolveGPU``)
or differentiates a forecast.  The cases cover those calls from the
reference's CPU configuration (ne = 6, nz = 10) to the full-size grid
(ne = 60, nz = 64), p = 3 and 4, both precisions, tracers, limited tracers,
forcing, terrain, columns taller than a wavefront and odd layer counts.

The grid, the states and ``exact`` are plain torch in this file; the library
is reached through its host module only.
"""
import importlib
import math
import os
import sys

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

if os.getcwd() not in sys.path:
    sys.path.insert(0, os.getcwd())
_pkg = importlib.import_module("__graft_entry__").load_package()
host, D = _pkg.host, _pkg.discretization

PHYS = D.Phys()
RAD, TOP = PHYS.RadEarth, 30000.0
DEV, F64 = "cuda", torch.float64
DAY = 86400.0


# ---------------------------------------------------------------- the cases
def _case(name, kind, ne, nz, p=4, steps=1, precision="fp64", ntr=0, limited=False, forcing=False, terrain=False,
          members=1):
    return dict(name=name, kind=kind, ne=ne, nz=nz, p=p, steps=steps, precision=precision, ntr=ntr, limited=limited,
                forcing=forcing, terrain=terrain, members=members)


def listed():
    return [
        # the reference's CPU configuration, one step per call: launches and host calls count
        _case("step_ne6_nz10", "step", 6, 10),
        # a Held-Suarez run at the reference's order 3, a layer count that no lane group divides
        _case("forced_ne30_p3_nz45", "run", 30, 45, p=3, steps=2, forcing=True),
        # the drop-in's configuration: an ordinary forecast segment
        _case("run_ne30_nz64", "run", 30, 64, steps=4),
        # the full-size grid, FP64 and mixed precision
        _case("run_ne60_nz64", "run", 60, 64, steps=4),
        _case("mixed_ne60_nz64", "run", 60, 64, precision="mixed"),
        # 32 ensemble members on grids of uneven size (ne 8, 12, 16), captured steps replayed
        _case("ensemble_32_nz32", "graph", 16, 32, steps=4, members=32),
        # an integrator of the caller's own: the tendency, and the column solve, as separate calls
        _case("tendency_ne30_nz64", "tendency", 30, 64),
        _case("column_ne30_nz64", "column", 30, 64),
        # two tracers, with the plain and with the limited horizontal transport
        _case("tracers_ne24_nz40", "run", 24, 40, steps=2, ntr=2),
        _case("limited_ne24_nz40", "run", 24, 40, steps=2, ntr=2, limited=True),
        # mountains, and columns taller than a wavefront
        _case("terrain_ne20_nz70", "run", 20, 70, steps=2, terrain=True),
        # a forecast's gradient with respect to its initial state (forward and reverse sweep)
        _case("gradient_ne16_nz32", "gradient", 16, 32, steps=12),
    ]


def draw(rng):
    """One more case: any call, any option that goes with it, sizes spread over the logarithm of the grid's points."""
    kind = rng.choice(["run"] * 5 + ["step", "graph", "tendency", "column", "gradient"])
    p = rng.choice([3, 4, 4])
    ne = int(round(math.exp(rng.uniform(math.log(4.0), math.log(40.0)))))
    nz = rng.choice([rng.randint(8, 64), rng.randint(8, 64), 32, 64, rng.randint(65, 90)])
    c = _case("", kind, ne, nz, p=p, steps=rng.randint(1, 4))
    if kind == "run":
        option = rng.choice(["plain", "plain", "mixed", "tracers", "limited", "forcing", "terrain"])
        if option == "mixed":
            c.update(precision="mixed", nz=min(nz, 64), steps=1)
        c.update(ntr=rng.randint(1, 3) if option in ("tracers", "limited") else 0, limited=option == "limited",
                 forcing=option == "forcing", terrain=option == "terrain")
        if option in ("tracers", "limited", "terrain") or nz > 64:
            c["steps"] = min(c["steps"], 2)
    elif kind == "graph":
        c.update(ne=min(ne, 16), nz=min(nz, 48), members=rng.randint(1, 16))
    elif kind == "gradient":
        c.update(ne=min(ne, 14), nz=min(nz, 40), steps=rng.randint(2, 6))
    del c["name"]
    return c


def _grids(case):
    """The ne of each member: the case's, or 8, 12, 16 of it in turn (at most the case's) for an ensemble."""
    ne, m = case["ne"], case["members"]
    return [ne] if m == 1 else [max(3, ne * (2 + k % 3) // 4) for k in range(m)]


def _dt(case):
    return min(300.0, 3000.0 / case["ne"])


# ---------------------------------------------------------------- the grid
_BASIS = {}


def _basis(p):
    """Gauss-Lobatto nodes and weights, DS[i,k] = l_k'(x_i) and DW = -W^-1 DS^T W (numpy)."""
    if p not in _BASIS:
        P = np.polynomial.legendre.Legendre.basis(p)
        x = np.concatenate([[-1.0], np.sort(P.deriv().roots().real), [1.0]])
        x = 0.5 * (x - x[::-1])
        w = 2.0 / (p * (p + 1) * P(x) ** 2)
        b = np.array([1.0 / np.prod(x[j] - np.delete(x, j)) for j in range(p + 1)])
        DS = np.array([[b[k] / b[i] / (x[i] - x[k]) if i != k else 0.0 for k in range(p + 1)] for i in range(p + 1)])
        DS -= np.diag(DS.sum(1))
        _BASIS[p] = x, w, DS, -(DS.T * w[None, :]) / w[:, None]
    return _BASIS[p]


def _panel_axes():
    """Six panels of the cube: the directions of the first and second coordinate and of the outer normal."""
    e = np.eye(3, dtype=np.int64)
    return [(e[1], e[2], e[0]), (-e[0], e[2], e[1]), (-e[1], e[2], -e[0]), (e[0], e[2], -e[1]), (e[1], -e[0], e[2]),
            (e[1], e[0], -e[2])]


def _surface(lam, lat):
    """A smooth surface height of a few ridges (m)."""
    return 800.0 * torch.cos(lat) ** 2 * (1.0 + torch.sin(2.0 * lam) * torch.cos(3.0 * lat)) ** 2 / 4.0


def _grid(ne, p, nz, terrain):
    """A Discretization on the GPU: equiangular cubed sphere, bilinear elements projected to the sphere, shallow metric."""
    N, NN = p + 1, (p + 1) ** 2
    x, w, DS, DW = _basis(p)
    NF = 6 * ne * ne
    axes = torch.as_tensor(np.array(_panel_axes()))
    k = torch.arange(ne)
    pan, ej, ei = (a.reshape(-1) for a in torch.meshgrid(torch.arange(6), k, k, indexing="ij"))
    # integer lattice of the nodes on the cube's surface (2 ne p wide): shared nodes have equal coordinates
    loc = torch.arange(N)
    I, J = loc.repeat(N), loc.repeat_interleave(N)
    a1 = 2 * (ei[:, None] * p + I[None]) - ne * p
    a2 = 2 * (ej[:, None] * p + J[None]) - ne * p
    A = axes[pan]
    pt = a1[..., None] * A[:, None, 0] + a2[..., None] * A[:, None, 1] + ne * p * A[:, None, 2]
    key = ((pt[..., 0] + ne * p) * (2 * ne * p + 1) + pt[..., 1] + ne * p) * (2 * ne * p + 1) + pt[..., 2] + ne * p
    ids, glob = torch.unique(key.to(DEV), return_inverse=True)
    num_g = int(ids.numel())
    # element corners on the sphere, then the bilinear map
    A, pan = A.to(DEV, F64), None
    tan = torch.tan(torch.linspace(-1.0, 1.0, ne + 1, dtype=F64) * (math.pi / 4.0))
    tan = 0.5 * (tan - tan.flip(0))
    tan[0], tan[-1] = -1.0, 1.0
    tan = tan.to(DEV)
    ei, ej = ei.to(DEV), ej.to(DEV)

    def corner(di, dj):
        c = tan[ei + di][:, None] * A[:, 0] + tan[ej + dj][:, None] * A[:, 1] + A[:, 2]
        return RAD * c / c.norm(dim=1, keepdim=True)

    C = [corner(0, 0), corner(1, 0), corner(1, 1), corner(0, 1)]
    xt = torch.as_tensor(x, device=DEV)
    xi, eta = xt[I.to(DEV)][None, :, None], xt[J.to(DEV)][None, :, None]
    wt = [(1 - xi) * (1 - eta), (1 + xi) * (1 - eta), (1 + xi) * (1 + eta), (1 - xi) * (1 + eta)]
    P = 0.25 * sum(f * c[:, None] for f, c in zip(wt, C))
    P1 = 0.25 * sum(f * c[:, None] for f, c in zip((-(1 - eta), 1 - eta, 1 + eta, -(1 + eta)), C))
    P2 = 0.25 * sum(f * c[:, None] for f, c in zip((-(1 - xi), -(1 + xi), 1 + xi, 1 - xi), C))
    r = P.norm(dim=2, keepdim=True)
    s = P / r + 0.0  # no negative zeros: the longitude of a pole is 0 in every element
    t1, t2 = (RAD * (q - s * (s * q).sum(2, keepdim=True)) / r for q in (P1, P2))
    lam, lat = torch.atan2(s[..., 1], s[..., 0]), torch.asin(s[..., 2].clamp(-1.0, 1.0))
    east = torch.stack([-lam.sin(), lam.cos(), torch.zeros_like(lam)], 2)
    north = torch.stack([-lat.sin() * lam.cos(), -lat.sin() * lam.sin(), lat.cos()], 2)
    L11, L12, L21, L22 = ((q * e).sum(2)[:, None, :, None] for q, e in
                          ((t1, east), (t2, east), (t1, north), (t2, north)))  # (NF, 1, NN, 1)
    # heights of the interfaces (terrain-following below 70 % of the top)
    z = torch.as_tensor(np.cumsum(np.concatenate([[0.0], np.full(nz, TOP / nz)])), device=DEV)
    if terrain:
        e = z / TOP
        low = torch.where(e <= 0.7, torch.sinh((0.7 - e) / 0.8 / 0.7) / math.sinh(1.0 / 0.8), torch.zeros_like(e))
        h = z[None, None] + _surface(lam, lat)[..., None] * low[None, None]
    else:
        h = z[None, None].expand(1, NN, nz + 1)
    hg = h.reshape(-1, N, N, nz + 1)  # (., J, I, interface)
    Dt = torch.as_tensor(DS, device=DEV)
    h1, h2 = torch.zeros_like(hg), torch.zeros_like(hg)
    for q in range(N):
        h1 = h1 + Dt[:, q][None, None, :, None] * hg[:, :, q:q + 1]
        h2 = h2 + Dt[:, q][None, :, None, None] * hg[:, q:q + 1]

    def both(f):  # interface values -> (., Nz, NN, K)
        f = f.reshape(-1, NN, nz + 1).permute(0, 2, 1)
        return torch.stack([f[:, :-1], f[:, 1:]], 3)

    hK, L31, L32 = both(hg), both(h1), both(h2)
    L33 = (0.5 * (hK[..., 1] - hK[..., 0]))[..., None]
    dX = torch.empty((NF, nz, NN, 2, 3, 3), dtype=F64, device=DEV)  # [..., j, i] = dXdxI[i, j]
    dX[..., 0, 0], dX[..., 0, 1], dX[..., 0, 2] = L22 * L33, -(L21 * L33), L21 * L32 - L22 * L31
    dX[..., 1, 0], dX[..., 1, 1], dX[..., 1, 2] = -(L12 * L33), L11 * L33, -(L11 * L32 - L12 * L31)
    dX[..., 2, 0], dX[..., 2, 1], dX[..., 2, 2] = 0.0, 0.0, L11 * L22 - L12 * L21
    jac = ((L11 * L22 - L12 * L21) * L33).expand(NF, nz, NN, 1)
    Jt = torch.empty((NF, nz, 2, NN), dtype=F64, device=DEV)
    Jt[:, :, 0], Jt[:, :, 1] = jac[..., 0], jac[..., 0]
    X = torch.empty((NF, nz, 3, 2, NN), dtype=F64, device=DEV)
    for q in range(3):
        X[:, :, q] = (s[..., q][:, None, :, None] * (RAD + hK)).permute(0, 1, 3, 2)
    # mass: sum of J over a node's copies, one copy after the other
    flat = glob.reshape(-1)
    order = torch.argsort(flat, stable=True)
    start = torch.searchsorted(flat[order], torch.arange(num_g, device=DEV))
    rank = torch.empty_like(flat)
    rank[order] = torch.arange(flat.numel(), device=DEV) - start[flat[order]]
    M = torch.zeros((2, num_g, nz), dtype=F64, device=DEV)
    Jn = jac[..., 0].permute(0, 2, 1).reshape(-1, nz)
    for q in range(int(rank.max()) + 1):
        c = torch.nonzero(rank == q).reshape(-1)
        M[0, flat[c]] += Jn[c]
    M[1] = M[0]
    dz = torch.empty((num_g, nz), dtype=F64, device=DEV)
    first = order[start]
    dz[:] = (hK[..., 1] - hK[..., 0]).expand(NF, nz, NN).permute(0, 2, 1).reshape(-1, nz)[first]
    disc = D.Discretization(ne=ne, p=p, nz=nz, H=TOP, rad=RAD, grid=None, glob=(glob + 1).contiguous(), num_g=num_g,
                            DS=DS, DW=DW, xw=x, w=w, z=None, dXdxI=dX, J=Jt, X=X, M=M, dz=dz)
    zm = (hK.mean(3)).expand(NF, nz, NN).permute(0, 2, 1).reshape(-1, nz)[first]
    return disc, torch.stack([lam.reshape(-1)[first], lat.reshape(-1)[first]], 1).contiguous(), zm


# ---------------------------------------------------------------- the state
def _state(lonlat, zm, ntr, seed):
    """A jet with a meridional wave, 1 K of potential-temperature noise, 0.1 m/s of noise in w, and tracers with steps."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))

    def noise():
        return 2.0 * torch.rand(zm.shape, generator=g, device=DEV, dtype=F64) - 1.0

    lam, lat = lonlat[:, :1], lonlat[:, 1:]
    T = 288.0 - 0.005 * zm
    pr = 1.0e5 * (T / 288.0) ** (PHYS.Grav / (PHYS.Rd * 0.005))
    rho = pr / (PHYS.Rd * T)
    theta = T * (PHYS.p0 / pr) ** PHYS.kappa + noise()
    taper = torch.cos(0.5 * math.pi * ((zm - 15000.0) / (TOP - 15000.0)).clamp(0.0, 1.0)) ** 2
    U = torch.empty((5 + ntr,) + tuple(zm.shape), dtype=F64, device=DEV)
    U[0] = rho
    U[1] = 35.0 * torch.sin(2.0 * lat) ** 2 * taper
    U[2] = 5.0 * torch.cos(lat) ** 2 * torch.sin(3.0 * lam) * taper
    U[3] = 0.1 * noise()
    U[3, :, -1] = 0.0
    U[4] = rho * theta
    for t in range(ntr):
        q = 1e-3 * (1.0 + ((lam > -1.0 + t) & (lam < 0.5 + t)).to(F64)) if t % 2 == 0 else 1e-3 * (1.5 + torch.sin(lam + t))
        U[5 + t] = rho * (q * (1.0 + 0.1 * noise()))
    return U


def _inputs(case, seed, ne=None, member=0):
    disc, lonlat, zm = _grid(ne or case["ne"], case["p"], case["nz"], case["terrain"])
    return disc, lonlat, _state(lonlat, zm, case["ntr"], 1000 * int(seed) + member)


def prepare(case, seed):
    kind = case["kind"]
    if case["members"] > 1:
        grids = {ne: _grid(ne, case["p"], case["nz"], False) for ne in sorted(set(_grids(case)))}
        ens = host.ensemble_setup([grids[ne][0] for ne in _grids(case)], PHYS, device=DEV, precision=case["precision"])
        V0 = torch.cat([_state(grids[ne][1], grids[ne][2], 0, 1000 * int(seed) + m)
                        for m, ne in enumerate(_grids(case))], 1).contiguous()
        FE, Metric, Global, Cache, JCache = ens.FE[0], ens.Metric[0], ens.Global, ens.Cache, ens.JCache
        ctx = Global._ctx
    else:
        disc, lonlat, V0 = _inputs(case, seed)
        FE, Metric, Global, Cache, JCache = host.device_setup(disc, PHYS, device=DEV, precision=case["precision"],
                                                              NumTr=case["ntr"])
        if case["limited"]:
            Global.Model.HorLimit = True
            FE.w = torch.as_tensor(disc.w, device=DEV)
        if case["forcing"]:
            Global.Model.Forcing = True
            Metric.xS = lonlat
        ctx = host.init_context(FE, Metric, PHYS, Global)
    st = dict(kind=kind, steps=case["steps"], dt=_dt(case), FE=FE, Metric=Metric, Global=Global, Cache=Cache,
              JCache=JCache, ctx=ctx, V0=V0, V=V0.clone())
    if kind == "graph":
        ctx.graph_create(st["V"], st["dt"], Cache, JCache, nsteps=case["steps"])
    elif kind == "tendency":
        st["F"] = torch.empty_like(V0)
        Global.dtauStage = st["dt"]
    elif kind == "column":
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        scale = torch.tensor([1e-6, 1e-4, 1e-4, 1e-4, 1e-3], dtype=F64, device=DEV)[:, None, None]
        st["fV"] = scale * torch.randn(V0.shape, generator=g, device=DEV, dtype=F64)
        st["fV"][3, :, -1] = 0.0
        st["k"], st["v"] = torch.zeros_like(V0), st["fV"].clone()
        host.FcnPrepareGPU(V0, FE, Metric, PHYS, Cache, None, Global, None, host.CompressibleShallow())
    elif kind == "gradient":
        st["every"] = 4
        st["work"] = ctx.adjoint_work(case["steps"], st["every"])
        st["Vf"] = torch.empty_like(V0)
    return st


def run(st):
    kind, dt, V, V0 = st["kind"], st["dt"], st["V"], st["V0"]
    FE, Metric, Global, Cache, JCache, ctx = (st[k] for k in ("FE", "Metric", "Global", "Cache", "JCache", "ctx"))
    eq = host.CompressibleShallow()
    if kind == "run":  # a forecast from the analysis
        V.copy_(V0)
        host.TimeStepper(V, dt, st["steps"], FE, Metric, PHYS, Cache, JCache, Global)
        return V
    if kind == "step":
        V.copy_(V0)
        host.RosenbrockSchur(V, dt, host.FcnGPU, host.FcnPrepareGPU, host.JacSchurGPU, FE, Metric, PHYS, Cache, JCache,
                             None, Global, None, eq)
        return V
    if kind == "graph":
        V.copy_(V0)
        ctx.graph_launch()
        return V
    if kind == "tendency":
        host.FcnPrepareGPU(V0, FE, Metric, PHYS, Cache, None, Global, None, eq)
        host.FcnGPU(st["F"], V0, FE, Metric, PHYS, Cache, None, Global, None, eq)
        return {"aux": Cache.AuxG[:3], "F": st["F"], "cache": Cache.Temp1}
    if kind == "column":
        st["v"].copy_(st["fV"])  # the solve overwrites its right-hand side
        JCache.CompTri = True
        host.JacSchurGPU(JCache, V0, FE, Metric, PHYS, Cache, Global, None, eq)
        host.SchurSolveGPU(st["k"], st["v"], JCache, dt, Cache, Global)
        return {"k": st["k"], "JRhoW": JCache.JRhoW, "JWRho": JCache.JWRho, "JWRhoTh": JCache.JWRhoTh,
                "JRhoThW": JCache.JRhoThW}
    # gradient of the sum over the lowest level of rho theta^2 after the steps
    Vf = st["Vf"]
    ctx.rw_forward_ckpt(V0, dt, st["steps"], st["every"], Vf, st["work"])
    lam = torch.zeros_like(V0)
    theta = Vf[4, :, 0] / Vf[0, :, 0]
    lam[4, :, 0] = 2.0 * theta
    lam[0, :, 0] = -theta * theta
    ctx.rw_adjoint_ckpt(dt, st["steps"], st["every"], lam, st["work"])
    return {"Vf": Vf, "gradient": lam}


def work(case):
    """Bytes: the state in and out, the mass, layer sizes and metric (5 words per element point on flat uniform layers, 17
    over terrain) once per step or call; operations: about 900 per element point and tendency, 100 per point and tracer."""
    n2, nz = (case["p"] + 1) ** 2, case["nz"]
    el = sum(6 * ne * ne * n2 * nz for ne in _grids(case))
    pts = sum((6 * ne * ne * case["p"] ** 2 + 2) * nz for ne in _grids(case))
    met = (17 if case["terrain"] else 5) * el
    nv = 5 + case["ntr"]
    fcn = (900.0 + 100.0 * case["ntr"]) * el
    if case["kind"] == "tendency":  # U -> p, T, theta, Temp1, F
        return {"bytes": 8.0 * ((5 + 2 + 3 + 5 + 5) * pts + met), "flops": fcn + 60.0 * pts}
    if case["kind"] == "column":  # rho, rho theta, dz, v -> J blocks, tri, k
        return {"bytes": 8.0 * (3 + 5 + 11 + 5) * pts, "flops": 300.0 * pts}
    step = {"bytes": 8.0 * ((2 * nv + 3) * pts + met), "flops": 3.0 * (fcn + 300.0 * pts)}
    n = case["steps"] * (3 if case["kind"] == "gradient" else 1)  # forward, and about twice that in reverse
    return {k: n * v for k, v in step.items()}


# ------------------------------------------------ the same in plain torch, 64 bits
class _Exact:
    def __init__(self, case, disc, lonlat):
        self.case, self.N = case, case["p"] + 1
        self.NF, self.NN, self.nz = disc.glob.shape[0], self.N ** 2, disc.nz
        self.glob = (disc.glob - 1).reshape(-1)
        self.num_g, self.dz, self.M = disc.num_g, disc.dz, disc.M
        self.D, self.DW = torch.as_tensor(disc.DS, device=DEV), torch.as_tensor(disc.DW, device=DEV)
        t = lambda a: a.permute(0, 2, 1).contiguous()  # noqa: E731  (NF, Nz, NN) -> (NF, NN, Nz)
        self.d = {(a, b, K): t(disc.dXdxI[:, :, :, K, b, a]) for a in range(3) for b in range(3) for K in range(2)
                  if not (a < 2 and b == 2)}
        self.J = [t(disc.J[:, :, K]) for K in range(2)]
        x = 0.5 * (disc.X[:, :, :, 0] + disc.X[:, :, :, 1])
        self.cor = t(2.0 * PHYS.Omega * x[:, :, 2] / x.norm(dim=2))
        self.S = {(a, b): self.d[a, b, 0] + self.d[a, b, 1] for a in range(2) for b in range(2)}
        self.Js = self.J[0] + self.J[1]
        self.Ms = self.M[0] + self.M[1]
        self.hyper = 5.0e14 * (30.0 / disc.ne) ** 3.2
        self.lat = lonlat[:, 1:]

    def g(self, f):  # global -> element nodes
        return f.index_select(0, self.glob).reshape(self.NF, self.NN, -1)

    def dss(self, f):  # element nodes -> sum over the copies
        z = torch.zeros((self.num_g, f.shape[2]), dtype=F64, device=DEV)
        return z.index_add(0, self.glob, f.reshape(-1, f.shape[2]))

    def dx(self, f, Dm=None):
        q = f.reshape(self.NF, self.N, self.N, -1)
        return torch.einsum("ik,fjkz->fjiz", self.D if Dm is None else Dm, q).reshape(f.shape)

    def dy(self, f, Dm=None):
        q = f.reshape(self.NF, self.N, self.N, -1)
        return torch.einsum("jk,fkiz->fjiz", self.D if Dm is None else Dm, q).reshape(f.shape)

    def pressure(self, U):
        return PHYS.p0 * torch.exp(torch.log(PHYS.Rd * U[4] / PHYS.p0) / (1.0 - PHYS.kappa))

    def scalar_lap(self, c, weight=None):
        S = self.S
        cx, cy = self.dx(c), self.dy(c)
        gx = (S[0, 0] * cx + S[1, 0] * cy) / self.Js
        gy = (S[0, 1] * cx + S[1, 1] * cy) / self.Js
        fx, fy = S[0, 0] * gx + S[0, 1] * gy, S[1, 0] * gx + S[1, 1] * gy
        if weight is not None:
            fx, fy = weight * fx, weight * fy
        return self.dx(fx, self.DW) + self.dy(fy, self.DW)

    def rot_grad(self, a, b, c, e):
        """Weak rot curl of (a, b) and grad div of (c, e)."""
        S = self.S
        curl = (self.dx(S[0, 0] * b - S[0, 1] * a) + self.dy(S[1, 0] * b - S[1, 1] * a)) / self.Js
        div = (self.dx(S[0, 0] * c + S[0, 1] * e) + self.dy(S[1, 0] * c + S[1, 1] * e)) / self.Js
        cx, cy, ex, ey = self.dx(curl, self.DW), self.dy(curl, self.DW), self.dx(div, self.DW), self.dy(div, self.DW)
        return (S[0, 1] * cx + S[1, 1] * cy, -S[0, 0] * cx - S[1, 0] * cy, S[0, 0] * ex + S[1, 0] * ey,
                S[0, 1] * ex + S[1, 1] * ey)

    def cache(self, U):
        r, u, v = self.g(U[0]), self.g(U[1]), self.g(U[2])
        a, b, c, e = self.rot_grad(u, v, u, v)
        out = [-a, -b, c, e, self.scalar_lap(self.g(U[4]) / r)]
        if not self.case["limited"]:
            out += [self.scalar_lap(self.g(U[k]) / r) for k in range(5, U.shape[0])]
        return torch.stack([self.dss(f) / self.Ms for f in out])

    @staticmethod
    def recon(cm, c, cp, cpp, Jm, J, Jp, Jpp):
        one = torch.ones_like(c)
        kR, kL = J / (J + Jp) * ((Jm + J) / (Jm + J + Jp)), J / (Jm + J) * (Jp / (Jm + J + Jp))
        r = (c - cm) / (cp - c + 1e-20)
        left = c + torch.relu(torch.minimum(r, torch.minimum(kL * r + kR, one))) * (cp - c)
        kL, kR = Jp / (Jp + J) * ((Jpp + Jp) / (J + Jp + Jpp)), Jp / (Jpp + Jp) * (J / (J + Jp + Jpp))
        r = (cp - cpp) / (c - cp + 1e-20)
        return left, cp + torch.relu(torch.minimum(r, torch.minimum(kR * r + kL, one))) * (c - cp)

    def tendency(self, U):
        d, S, hd, nz = self.d, self.S, self.hyper, self.nz
        C, p = self.cache(U), self.g(self.pressure(U))
        r, u, v, wh = (self.g(U[k]) for k in range(4))
        lo, up = (lambda f: f[..., :-1]), (lambda f: f[..., 1:])
        bottom = -(d[2, 0, 0] * u + d[2, 1, 0] * v)[..., :1] / d[2, 2, 0][..., :1]
        wl = torch.cat([bottom, lo(wh)], 2)
        f = [0.0] * U.shape[0]
        # hyperviscosity of the cache
        a, b, c, e = self.rot_grad(self.g(C[0]), self.g(C[1]), self.g(C[2]), self.g(C[3]))
        f[1], f[2] = hd * (a - c), hd * (b - e)
        # momentum
        w = [wl, wh]
        tu = [d[2, 2, K] * v - d[2, 1, K] * w[K] for K in range(2)]
        tv = [d[2, 2, K] * u - d[2, 0, K] * w[K] for K in range(2)]
        tw = [d[2, 1, K] * u - d[2, 0, K] * v for K in range(2)]
        zero = torch.zeros_like(u[..., :1])
        flux = [0.5 * (up(t[0]) - lo(t[1])) for t in (tu, tv, tw)]
        fl = [torch.cat([zero, q], 2) for q in flux]  # through the lower interface
        fu = [torch.cat([q, zero], 2) for q in flux]  # through the upper interface
        FU = -v * (fl[2] + fu[2]) - wl * fl[1] - wh * fu[1] + v * self.cor * self.Js
        FV = u * (fl[2] + fu[2]) - wl * fl[0] - wh * fu[0] - u * self.cor * self.Js
        FW = [u * fl[1] + v * fl[0], u * fu[1] + v * fu[0]]
        Uk, Vk, Wk = [], [], []
        for K in range(2):
            Uk.append(0.5 * (tu[1] - tu[0]) - self.dx(d[0, 1, K] * w[K]) - self.dy(d[1, 1, K] * w[K]))
            Vk.append(0.5 * (tv[1] - tv[0]) - self.dx(d[0, 0, K] * w[K]) - self.dy(d[1, 0, K] * w[K]))
            Wk.append(0.5 * (tw[1] - tw[0]) + self.dx(d[0, 1, K] * u - d[0, 0, K] * v) +
                      self.dy(d[1, 1, K] * u - d[1, 0, K] * v))
        f[1] = f[1] - v * (Wk[0] + Wk[1]) - wl * Vk[0] - wh * Vk[1] + FU
        f[2] = f[2] + u * (Wk[0] + Wk[1]) - wl * Uk[0] - wh * Uk[1] + FV
        mw = [r * (u * Vk[K] + v * Uk[K] + FW[K]) for K in range(2)]
        # kinetic energy, pressure, gravity
        kin = [0.5 * (u * u + v * v) + 0.5 * w[K] * w[K] for K in range(2)]
        jump = 0.5 * (up(kin[0]) - lo(kin[1]))
        gz = [torch.cat([zero, jump], 2) + 0.5 * (kin[1] - kin[0]), torch.cat([jump, zero], 2) + 0.5 * (kin[1] - kin[0])]
        px, py = self.dx(p), self.dy(p)
        hyd = -PHYS.Grav * r * self.Js / (d[2, 2, 0] + d[2, 2, 1])
        for q in range(2):
            pg = S[0, q] * px + S[1, q] * py + hyd * (d[2, q, 0] + d[2, q, 1])
            kg = sum(-(d[0, q, K] * self.dx(kin[K]) + d[1, q, K] * self.dy(kin[K])) - gz[K] * d[2, q, K]
                     for K in range(2))
            f[1 + q] = f[1 + q] + kg - pg / r
        mw = [mw[K] - r * gz[K] * d[2, 2, K] for K in range(2)]
        bal = -(0.5 * (up(p) - lo(p)) * (lo(d[2, 2, 1]) + up(d[2, 2, 0])) +
                PHYS.Grav * (lo(r) * lo(self.J[1]) + up(r) * up(self.J[0])))
        fw = lo(mw[1]) + up(mw[0]) + bal
        # mass, theta and tracer transport
        wcon = lo(r) * lo(d[2, 0, 1] * u + d[2, 1, 1] * v + d[2, 2, 1] * wh) + \
            up(r) * (up(d[2, 0, 0] * u + d[2, 1, 0] * v) + up(d[2, 2, 0]) * lo(wh))
        mx, my = -r * (S[0, 0] * u + S[0, 1] * v), -r * (S[1, 0] * u + S[1, 1] * v)
        pad = lambda q: torch.cat([zero, q], 2) - torch.cat([q, zero], 2)  # noqa: E731
        f[0] = self.dx(mx) + self.dy(my) + pad(0.5 * wcon)
        low = lambda q: torch.cat([q[..., :1], q[..., :-2]], 2)  # noqa: E731
        high = lambda q: torch.cat([q[..., 2:], q[..., -1:]], 2)  # noqa: E731
        Jq = [low(self.Js), lo(self.Js), up(self.Js), high(self.Js)]
        for k in [4] + ([] if self.case["limited"] else list(range(5, U.shape[0]))):
            c = self.g(U[k]) / r
            left, right = self.recon(low(c), lo(c), up(c), high(c), *Jq)
            fl = 0.25 * ((wcon.abs() + wcon) * left + (-wcon.abs() + wcon) * right)
            f[k] = self.dx(mx * c) + self.dy(my * c) + pad(fl) - hd * self.scalar_lap(self.g(C[k]), r)
        F = [self.dss(q) / self.Ms if k != 3 and isinstance(q, torch.Tensor) else None for k, q in enumerate(f)]
        den = U[0][:, 1:] * self.M[0][:, 1:] + U[0][:, :-1] * self.M[1][:, :-1]
        F[3] = torch.cat([self.dss(fw) / den, torch.zeros_like(den[:, :1])], 1)
        F = torch.stack([q if q is not None else torch.zeros_like(U[0]) for q in F])
        if self.case["forcing"]:
            F = F + self.forcing(U)
        return F, C

    def forcing(self, U):
        hs = dict(k_a=1.0 / (40.0 * DAY), k_f=1.0 / DAY, k_s=1.0 / (4.0 * DAY), DeltaT_y=60.0, DeltaTh_z=10.0,
                  T_equator=315.0, T_min=200.0, sigma_b=0.7)
        p = self.pressure(U)
        sig = p / PHYS.p0
        hf = torch.relu((sig - hs["sigma_b"]) / (1.0 - hs["sigma_b"]))
        kT = torch.where(sig < 0.7, hs["k_a"] + (hs["k_s"] - hs["k_a"]) * hf * self.lat.cos() ** 4, 0.0 * sig)
        eq = (hs["T_equator"] - hs["DeltaT_y"] * self.lat.sin() ** 2 -
              hs["DeltaTh_z"] * torch.log(sig) * self.lat.cos() ** 2) * sig ** PHYS.kappa
        dT = kT * (p / (U[0] * PHYS.Rd) - eq.clamp(min=hs["T_min"]))
        G = torch.zeros_like(U)
        G[1], G[2], G[4] = -hs["k_f"] * hf * U[1], -hs["k_f"] * hf * U[2], -U[0] * dT / sig ** PHYS.kappa
        return G

    def jacobian(self, U):
        lo, up = (lambda f: f[:, :-1]), (lambda f: f[:, 1:])
        r, t, z = U[0], U[4], self.dz
        dp = PHYS.Rd * (PHYS.Rd * t / PHYS.p0) ** (PHYS.kappa / (1.0 - PHYS.kappa))
        s = lo(z) + up(z)
        rf, tf = (lo(r) * lo(z) + up(r) * up(z)) / s, (lo(t) * lo(z) + up(t) * up(z)) / s
        return dict(rw=(-rf / lo(z), rf / up(z)), wt=(-up(dp) / rf * 2.0 / s, lo(dp) / rf * 2.0 / s),
                    wr=(-PHYS.Grav * up(z) / rf / s, -PHYS.Grav * lo(z) / rf / s), tw=(-tf / lo(z), tf / up(z)))

    def schur(self, v, J, fac):
        rw, wr, wt, tw = J["rw"], J["wr"], J["wt"], J["tw"]
        n = self.nz - 1
        diag = 1.0 / fac ** 2 - wr[1] * rw[0] - wr[0] * rw[1] - wt[1] * tw[0] - wt[0] * tw[1]
        upper = -wr[0][:, :-1] * rw[0][:, 1:] - wt[0][:, :-1] * tw[0][:, 1:]  # row i, column i+1
        lower = -wr[1][:, 1:] * rw[1][:, :-1] - wt[1][:, 1:] * tw[1][:, :-1]  # row i+1, column i
        rhs = v[3][:, :-1] / fac + wr[1] * v[0][:, :-1] + wr[0] * v[0][:, 1:] + wt[1] * v[4][:, :-1] + wt[0] * v[4][:, 1:]
        b, y = [diag[:, 0]], [rhs[:, 0]]
        for i in range(1, n):
            q = lower[:, i - 1] / b[-1]
            b.append(diag[:, i] - q * upper[:, i - 1])
            y.append(rhs[:, i] - q * y[-1])
        x = [y[-1] / b[-1]]
        for i in range(n - 2, -1, -1):
            x.append((y[i] - upper[:, i] * x[-1]) / b[i])
        kw = torch.stack(x[::-1], 1)
        zero = torch.zeros_like(kw[:, :1])
        add = lambda m: torch.cat([m[0] * kw, zero], 1) + torch.cat([zero, m[1] * kw], 1)  # noqa: E731
        k = [fac * (v[0] + add(rw)), fac * v[1], fac * v[2], torch.cat([kw, zero], 1), fac * (v[4] + add(tw))]
        # the lid row is not part of the system and has no tendency
        return torch.stack(k + [fac * v[q] for q in range(5, v.shape[0])])

    def step(self, Vn, dt):
        a, c, m = ((), (1.0,), (0.25, 0.25)), ((), (0.0,), (-0.75, -0.75)), (2.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0)
        J, k = self.jacobian(Vn), []
        for i in range(3):
            V = Vn + sum(a[i][j] * k[j] for j in range(i))
            f = self.tendency(V)[0] + sum(c[i][j] / dt * k[j] for j in range(i))
            k.append(self.schur(f, J, dt))
        return Vn + sum(m[i] * k[i] for i in range(3))


def exact(case, seed):
    dt, kind = _dt(case), case["kind"]
    if case["members"] > 1:
        grids = {ne: _grid(ne, case["p"], case["nz"], False) for ne in sorted(set(_grids(case)))}
        out = []
        for m, ne in enumerate(_grids(case)):
            E, V = _Exact(case, grids[ne][0], grids[ne][1]), _state(grids[ne][1], grids[ne][2], 0, 1000 * int(seed) + m)
            for _ in range(case["steps"]):
                V = E.step(V, dt)
            out.append(V)
        return torch.cat(out, 1)
    disc, lonlat, V0 = _inputs(case, seed)
    E = _Exact(case, disc, lonlat)
    if kind == "tendency":
        F, C = E.tendency(V0)
        p = E.pressure(V0)
        T = p / (PHYS.Rd * V0[0])
        return {"aux": torch.stack([p, T, (PHYS.p0 / p) ** PHYS.kappa * T]), "F": F, "cache": C}
    if kind == "column":
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        scale = torch.tensor([1e-6, 1e-4, 1e-4, 1e-4, 1e-3], dtype=F64, device=DEV)[:, None, None]
        v = scale * torch.randn(V0.shape, generator=g, device=DEV, dtype=F64)
        v[3, :, -1] = 0.0
        J = E.jacobian(V0)
        return {"k": E.schur(v, J, dt), **{name: torch.stack(J[q], 2) for name, q in
                (("JRhoW", "rw"), ("JWRho", "wr"), ("JWRhoTh", "wt"), ("JRhoThW", "tw"))}}
    if kind == "gradient":
        V0.requires_grad_(True)
        V = V0
        for _ in range(case["steps"]):
            V = checkpoint(E.step, V, dt, use_reentrant=False)
        (V[4, :, 0] ** 2 / V[0, :, 0]).sum().backward()
        return {"Vf": V.detach(), "gradient": V0.grad}
    if case["limited"]:
        return None  # the limiter's bounded iteration has no plain counterpart here
    V = V0
    for _ in range(case["steps"]):
        V = E.step(V, dt)
    return V
