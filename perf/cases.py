"""Timed cases: what a user of flurrypp_amd has it do, through its public entry points.

The cases are the steps that the package's own workloads take (flurrypp_amd.cases, bench.py, the
serving and batching loops), over the range of meshes, orders and precisions these run at:

* ``steps``   Solver.update(n): the RK loop of one case (Euler or Navier-Stokes, 2-D or 3-D, FP64 or
              mixed precision, fixed or CFL time step);
* ``monitor`` one iteration of the main loop with its residual monitor: update(1), dt, residual_norm;
* ``pmg``     one iteration of a steady solve: update(1) and a P-multigrid cycle;
* ``batch``   one step of a BatchedSolver over several channels of mixed orders, with multigrid;
* ``members`` one RK44 step driven through the solver's members one by one (calcResidual, timeStepA/B).

``exact`` computes the same outputs with plain torch in 64 bits, from the scheme's definition: flux
reconstruction on tensor-product Gauss points, DG correction, Rusanov/Roe and LDG common fluxes.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from flurrypp_amd import _native as nat
from flurrypp_amd import cases as workloads
from flurrypp_amd.batch import BatchedSolver, Member
from flurrypp_amd.solver import MultiGrid, Solver

GAMMA = 1.4
CFL_LIMIT = {0: 1.393, 1: 0.464, 2: 0.235, 3: 0.1453, 4: 0.100, 5: 0.0736}
MESH_SEED = 20261202
TGV_MACH, TGV_RE, TGV_PR = 0.1, 1600.0, 0.71
VORTEX_MACH, VORTEX_BETA = 0.5, 5.0


# ---------------------------------------------------------------------------
# the cases

def listed():
    return [
        # the smallest call: one step of the 8x8 vortex that the smoke run takes, latency alone
        dict(name="vortex2d_8_p3_step", do="steps", kind="vortex2d", n=8, order=3, steps=1, path="fp64", tuned=False),
        # the 2-D isentropic vortex at its full size: many short kernels
        dict(name="vortex2d_32_p3_20steps", do="steps", kind="vortex2d", n=32, order=3, steps=20, path="fp64",
             tuned=True),
        # a steady channel request of the served mix: update and multigrid cycle, ragged mesh
        dict(name="bump2d_67x29_p4_pmg", do="pmg", kind="bump2d", nx=67, ny=29, order=4, mach=0.35, path="fp64"),
        # the same in mixed precision, as half of the served requests start
        dict(name="bump2d_113x41_p3_pmg_mixed", do="pmg", kind="bump2d", nx=113, ny=41, order=3, mach=0.25,
             path="mixed"),
        # a step of the batched form: channels of orders 1 to 5, merged per order, with multigrid
        dict(name="batch_15_channels_pmg", do="batch", kind="bump2d", members=15, mesh_seed=7, path="fp64"),
        # unsteady served requests: the 3-D Euler vortex, global CFL step, FP64 and mixed, ragged sizes
        dict(name="vortex3d_17_p2_10steps", do="steps", kind="vortex3d", n=17, order=2, steps=10, path="fp64",
             tuned=False),
        dict(name="vortex3d_23_p4_4steps", do="steps", kind="vortex3d", n=23, order=4, steps=4, path="mixed",
             tuned=False),
        # the headline run: Navier-Stokes Taylor-Green vortex 48^3 P3, FP64, tuned as bench.py tunes it
        dict(name="tgv3d_ns_48_p3_4steps", do="steps", kind="tgv3d", n=48, order=3, viscous=True, steps=4, path="fp64",
             tuned=True),
        # its mixed-precision form
        dict(name="tgv3d_ns_40_p3_mixed_4steps", do="steps", kind="tgv3d", n=40, order=3, viscous=True, steps=4,
             path="mixed", tuned=True),
        # another order, a mesh that divides nothing
        dict(name="tgv3d_ns_37_p2_4steps", do="steps", kind="tgv3d", n=37, order=2, viscous=True, steps=4, path="fp64",
             tuned=True),
        # the main loop of an input-file run with its monitor at every iteration, default settings
        dict(name="tgv3d_ns_21_p4_monitor", do="monitor", kind="tgv3d", n=21, order=4, viscous=True, path="fp64",
             tuned=False),
        # a host program that drives its own RK loop through the solver's members
        dict(name="tgv3d_ns_18_p3_members", do="members", kind="tgv3d", n=18, order=3, viscous=True, path="staged",
             tuned=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["vortex2d", "vortex3d", "tgv3d", "tgv3d", "pmg", "batch", "monitor", "members"])
    path = "mixed" if rng.random() < 0.3 else "fp64"
    if kind == "vortex2d":
        return dict(do="steps", kind="vortex2d", n=_log_int(rng, 6, 96), order=rng.randint(1, 5),
                    steps=_log_int(rng, 1, 20), path=path, tuned=rng.random() < 0.5,
                    riemann=1 if rng.random() < 0.3 else 0)
    if kind == "vortex3d":
        P = rng.randint(2, 4)
        return dict(do="steps", kind="vortex3d", n=_log_int(rng, 8, {2: 40, 3: 34, 4: 26}[P]), order=P,
                    steps=rng.randint(1, 4), path=path, tuned=rng.random() < 0.5)
    if kind == "tgv3d":
        P = rng.randint(1, 5)
        return dict(do="steps", kind="tgv3d", n=_log_int(rng, 5, {1: 56, 2: 44, 3: 40, 4: 28, 5: 24}[P]), order=P,
                    viscous=rng.random() < 0.7, steps=rng.randint(1, 4), path=path, tuned=rng.random() < 0.5)
    if kind == "pmg":
        return dict(do="pmg", kind="bump2d", nx=_log_int(rng, 16, 128), ny=_log_int(rng, 8, 48),
                    order=rng.randint(1, 5), mach=round(rng.uniform(0.2, 0.5), 3), path=path)
    if kind == "batch":
        return dict(do="batch", kind="bump2d", members=rng.randint(4, 15), mesh_seed=rng.randint(1, 1000),
                    path="fp64")
    if kind == "monitor":
        P = rng.randint(1, 4)
        return dict(do="monitor", kind="tgv3d", n=_log_int(rng, 5, {1: 40, 2: 32, 3: 28, 4: 22}[P]), order=P,
                    viscous=rng.random() < 0.7, path="fp64", tuned=rng.random() < 0.5)
    P = rng.randint(1, 4)
    return dict(do="members", kind="tgv3d", n=_log_int(rng, 5, {1: 32, 2: 24, 3: 18, 4: 14}[P]), order=P,
                viscous=rng.random() < 0.7, path="staged", tuned=False)


def _channels(case):
    """(nx, ny, order, Mach) of the members of a batch: the ranges of the batched workload."""
    rng = np.random.default_rng(case["mesh_seed"])
    return [(int(rng.integers(16, 129)), int(rng.integers(8, 49)), 1 + i % 5, float(rng.uniform(0.2, 0.5)))
            for i in range(case["members"])]


def _box(case):
    """Dimension, elements per side, lower corner and side of a periodic box case."""
    if case["kind"] == "vortex2d":
        return 2, case["n"], -5.0, 10.0
    if case["kind"] == "vortex3d":
        return 3, case["n"], -5.0, 10.0
    return 3, case["n"], 0.0, 2.0 * math.pi


def _tgv_dt(case):
    """A fixed step at half the CFL limit of the initial field (wave speed |v| + c)."""
    return 0.5 * CFL_LIMIT[case["order"]] * (2.0 * math.pi / case["n"]) / (3.0 * (1.0 + 1.0 / TGV_MACH))


@functools.lru_cache(maxsize=3)
def _host_setup(kind, n, order, viscous, riemann, dt):
    """Mesh, operators and metric terms, which a program sets up once for all of its runs."""
    if kind == "vortex2d":
        return workloads.vortex2d(n=n, order=order, riemann=riemann)[0]
    if kind == "vortex3d":
        return workloads.vortex3d(n=n, order=order)[0]
    return workloads.tgv3d(n=n, order=order, viscous=1 if viscous else 0, dt=dt)[0]


@functools.lru_cache(maxsize=16)
def _channel_setup(nx, ny, order, mach):
    return workloads.bump2d(nx=nx, ny=ny, order=order, mach=mach, seed=MESH_SEED, time_type=6, cfl=0.9)[0]


# ---------------------------------------------------------------------------
# initial states, from the positions of the solution points

def _vortex_state(pos, seed, dims):
    """The isentropic vortex, its centre drawn from the seed, wrapped into the periodic box."""
    rng = np.random.default_rng(seed)
    cx, cy = rng.uniform(-2.0, 2.0, 2)
    x = np.mod(pos[..., 0] - cx + 5.0, 10.0) - 5.0
    y = np.mod(pos[..., 1] - cy + 5.0, 10.0) - 5.0
    f, eps, g = 1.0 - (x * x + y * y), VORTEX_BETA, GAMMA
    rho = np.maximum(np.power(1.0 - eps * eps * (g - 1.0) / (8.0 * g * math.pi ** 2) * np.exp(f), 1.0 / (g - 1.0)),
                     1e-3)
    vx = VORTEX_MACH * math.sqrt(g) - eps * y / (2.0 * math.pi) * np.exp(f / 2.0)
    vy = eps * x / (2.0 * math.pi) * np.exp(f / 2.0)
    U = np.zeros(pos.shape[:2] + (dims + 2,))
    U[..., 0], U[..., 1], U[..., 2] = rho, rho * vx, rho * vy
    U[..., -1] = np.power(rho, g) / (g - 1.0) + 0.5 * rho * (vx * vx + vy * vy)
    return U


def _tgv_state(pos, seed):
    """The Taylor-Green field, its phases drawn from the seed."""
    x, y, z = (pos[..., d] + s for d, s in enumerate(np.random.default_rng(seed).uniform(0.0, 2.0 * math.pi, 3)))
    u, v = np.sin(x) * np.cos(y) * np.cos(z), -np.cos(x) * np.sin(y) * np.cos(z)
    p = 1.0 / (GAMMA * TGV_MACH ** 2) + (np.cos(2 * x) + np.cos(2 * y)) * (np.cos(2 * z) + 2.0) / 16.0
    U = np.zeros(pos.shape[:2] + (5,))
    U[..., 0], U[..., 1], U[..., 2] = 1.0, u, v
    U[..., 4] = p / (GAMMA - 1.0) + 0.5 * (u * u + v * v)
    return U


def _channel_state(pos, mach, seed):
    """The free stream with a smooth disturbance of one per cent, a solve under way."""
    rng = np.random.default_rng(seed)
    x, y = pos[..., 0], pos[..., 1]
    a, ph = rng.uniform(-0.01, 0.01, 3), rng.uniform(0.0, 2.0 * math.pi, 3)
    rho = 1.0 + a[0] * np.sin(2.0 * x + ph[0]) * np.cos(3.0 * y)
    vx = mach * (1.0 + a[1] * np.sin(3.0 * x + ph[1]))
    vy = mach * a[2] * np.sin(2.0 * y + x + ph[2])
    p = (1.0 / GAMMA) * np.power(rho, GAMMA)
    U = np.zeros(pos.shape[:2] + (4,))
    U[..., 0], U[..., 1], U[..., 2] = rho, rho * vx, rho * vy
    U[..., 3] = p / (GAMMA - 1.0) + 0.5 * rho * (vx * vx + vy * vy)
    return U


def _initial(case, pos, seed):
    if case["kind"] == "bump2d":
        return _channel_state(pos, case["mach"], seed)
    if case["kind"] == "tgv3d":
        return _tgv_state(pos, seed)
    return _vortex_state(pos, seed, pos.shape[2])


# ---------------------------------------------------------------------------
# preparation and one pass

class _DeviceArray:
    """Device memory that belongs to `owner`: a tensor over it holds this object, and so its owner."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr="<f8", version=2)


def _view(owner, name, shape, step=0):
    """One of a context's arrays as a torch tensor, without a copy (fhip_device_ptr)."""
    p = ctypes.c_void_p()
    nat.hip_check(nat.hip_lib().fhip_device_ptr(owner._ctx, nat.ARR[name], step, ctypes.byref(p)))
    return torch.as_tensor(_DeviceArray(owner, p.value, shape), device="cuda")


PATHS = {"fp64": nat.PATH_FUSED, "mixed": nat.PATH_MIXED, "staged": nat.PATH_STAGED}


def prepare(case, seed):
    path = PATHS[case["path"]]
    if case["do"] == "batch":
        members = []
        for i, (nx, ny, order, mach) in enumerate(_channels(case)):
            setup = _channel_setup(nx, ny, order, mach)
            members.append(Member(setup, _channel_state(setup.geo.pos_spts, mach, seed * 1000 + i), (nx, ny, order)))
        batch = BatchedSolver(members, path=path, pmg=True, low_order=0, smooth_steps=2, autotune=True)
        views = {"P%d" % g.m.order: _view(g, "U_spts", g.m.U.shape) for g in batch.groups}
        return dict(case=case, batch=batch, views=views)
    if case["kind"] == "bump2d":
        setup = _channel_setup(case["nx"], case["ny"], case["order"], case["mach"])
    else:
        dt = _tgv_dt(case) if case["kind"] == "tgv3d" else None
        setup = _host_setup(case["kind"], case["n"], case["order"], case.get("viscous", False),
                            case.get("riemann", 0), dt)
    solver = Solver(setup.params, setup=setup)
    solver.initializeSolution(_initial(case, setup.geo.pos_spts, seed))
    state = dict(case=case, solver=solver, path=path, views={"U": _view(solver, "U_spts", solver.shape_spts)})
    if case["do"] == "pmg":
        state["mg"] = MultiGrid(solver, low_order=0, smooth_steps=2)
    if case["do"] == "members":
        state["views"]["divF"] = _view(solver, "divF_spts", solver.shape_spts, 3)
    if case.get("tuned"):
        solver.autotune(path)
    return state


def run(state):
    case, out = state["case"], dict(state["views"])
    if case["do"] == "batch":
        state["batch"].step(1)
        return out
    s = state["solver"]
    if case["do"] == "steps":
        s.update(case["steps"], path=state["path"])
    elif case["do"] == "pmg":
        s.update(1, path=state["path"], sync=False)
        state["mg"].cycle(state["path"])
    elif case["do"] == "monitor":
        s.update(1)
        out["dt"] = s.dt
        out["residual"] = s.residual_norm()
    else:
        p = s.params
        s.copyUspts_U0()
        for step in range(3):
            s.calcResidual(step)
            s.timeStepA(step, p.RKa[step + 1])
        s.calcResidual(3)
        s.copyU0_Uspts()
        for step in range(4):
            s.timeStepB(step)
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _stage(D, P, E, viscous, real):
    """Bytes and operations of one RK stage over E elements: the state read (and the step's start),
    the new state written, the metric terms and normals read; tensor-product operators, point and
    face fluxes."""
    P1, N = P + 1, D + 2
    S, F = P1 ** D, 2 * D * P1 ** (D - 1)
    nbytes = E * (3 * 8 * S * N + 8 * S + real * (S * D * D + F * (D + 1)))
    ops = S * N * 2 * D * P1 + 2 * F * N * 2 * P1 + S * N * 2 * 2 * D + S * N * (2 * D * D + 6) + F * 60
    if viscous:
        ops += S * N * (2 * D * P1 + 2 * 2 * D + 2 * D * D) + F * D * N * 2 * P1 + (S + F) * 120
    return nbytes, E * ops


def work(case):
    real = 4 if case["path"] == "mixed" else 8
    todo = []  # (D, P, E, viscous, stages)
    if case["kind"] == "bump2d":
        meshes = _channels(case) if case["do"] == "batch" else [(case["nx"], case["ny"], case["order"], 0)]
        for nx, ny, order, _ in meshes:
            todo.append((2, order, nx * ny, False, 5))  # the update and the fine residual of the cycle
            todo += [(2, q, nx * ny, False, 2 * 2 * 4 + 1) for q in range(order)]
    else:
        D, n, _, _ = _box(case)
        todo.append((D, case["order"], n ** D, bool(case.get("viscous")), 4 * case.get("steps", 1)))
    nbytes = flops = 0
    for D, P, E, viscous, stages in todo:
        b, f = _stage(D, P, E, viscous, real)
        nbytes, flops = nbytes + b * stages, flops + f * stages
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _lagrange(x, y):
    """[len(y)][len(x)] values of the Lagrange polynomials on x at y."""
    return np.array([[np.prod([(b - x[j]) / (x[i] - x[j]) for j in range(len(x)) if j != i]) for i in range(len(x))]
                     for b in y])


def _derivative(x):
    """[i][m] derivative of Lagrange polynomial m at node i."""
    n = len(x)
    w = np.array([np.prod([x[i] - x[j] for j in range(n) if j != i]) for i in range(n)])
    d = np.zeros((n, n))
    for i in range(n):
        for m in range(n):
            if i != m:
                d[i, m] = w[i] / (w[m] * (x[i] - x[m]))
        d[i, i] = -d[i].sum()
    return d


# faces of the reference element: dimension and side of the normal, and for each further dimension in
# the points' order whether it runs backwards
_FACES = {2: [(1, -1, [(0, 1)]), (0, 1, [(1, 1)]), (1, 1, [(0, -1)]), (0, -1, [(1, -1)])],
          3: [(2, -1, [(0, 1), (1, 1)]), (2, 1, [(0, -1), (1, 1)]), (0, -1, [(1, 1), (2, 1)]),
              (0, 1, [(1, -1), (2, 1)]), (1, -1, [(0, -1), (2, 1)]), (1, 1, [(0, 1), (2, 1)])]}


class _Scheme:
    """Operators of one order, geometry and neighbours of one structured mesh, and the residual."""

    def __init__(self, D, order, corners, neighbours, bc=None, viscous=False, riemann=0):
        """corners [E][2^D][D] in the elements' vertex order; neighbours [2D][E] element across each
        face (-1 on a boundary); bc [2D][E] boundary number (1 characteristic, 8 slip wall)."""
        dev = _device()
        self.D, self.P, self.viscous, self.riemann = D, order, viscous, riemann
        P1 = order + 1
        x, w = np.polynomial.legendre.leggauss(P1)
        leg = np.polynomial.legendre.Legendre
        dl, dr = leg.basis(order).deriv(), leg.basis(order + 1).deriv()
        edge = {1: 0.5 * (dl(x) + dr(x)), -1: 0.5 * (-1.0) ** order * (dl(x) - dr(x))}
        edge[-1] = -edge[-1]
        ends = {1: _lagrange(x, [1.0])[0], -1: _lagrange(x, [-1.0])[0]}
        S = P1 ** D
        coord = np.array([[s // P1 ** d % P1 for d in range(D)] for s in range(S)])
        d1 = _derivative(x)
        grad = np.zeros((D, S, S))
        for d in range(D):
            same = np.all(np.delete(coord[:, None], d, 2) == np.delete(coord[None], d, 2), axis=2)
            grad[d] = np.where(same, d1[coord[:, d][:, None], coord[:, d][None]], 0.0)
        to_f, corr, tn, ref, wf, partner = [], [], [], [], [], []
        for dim, side, tang in _FACES[D]:
            for q in range(P1 ** (D - 1)):
                at = [q // P1 ** t % P1 if s > 0 else order - q // P1 ** t % P1 for t, (_, s) in enumerate(tang)]
                on = np.all([coord[:, d] == a for (d, _), a in zip(tang, at)], axis=0)
                to_f.append(np.where(on, ends[side][coord[:, dim]], 0.0))
                corr.append(np.where(on, edge[side][coord[:, dim]], 0.0))
                tn.append([side if d == dim else 0 for d in range(D)])
                p = np.zeros(D)
                p[dim] = side
                for (d, _), a in zip(tang, at):
                    p[d] = x[a]
                ref.append(p)
                wf.append(np.prod([w[a] for a in at]))
                partner.append((dim, -side, tuple(sorted(zip([d for d, _ in tang], at)))))
        key = {}
        f = 0
        for dim, side, tang in _FACES[D]:
            for q in range(P1 ** (D - 1)):
                at = [q // P1 ** t % P1 if s > 0 else order - q // P1 ** t % P1 for t, (_, s) in enumerate(tang)]
                key[(dim, side, tuple(sorted(zip([d for d, _ in tang], at))))] = f
                f += 1
        t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=dev)  # noqa: E731
        self.points = x
        self.to_f, self.grad, self.corr, self.tn = t(to_f), t(grad), t(np.array(corr).T), t(tn)
        self.w_face = t(wf)
        self.w = t(np.prod([w[coord[:, d]] for d in range(D)], axis=0))
        # opposite flux point of the neighbour
        Ff, E = P1 ** (D - 1), corners.shape[0]
        nb = torch.as_tensor(np.repeat(neighbours, Ff, axis=0), device=dev)
        across = torch.as_tensor([key[p] for p in partner], device=dev)
        self.boundary = nb < 0
        self.across = across[:, None] * E + torch.where(self.boundary, torch.zeros_like(nb), nb)
        self.first = (nb > torch.arange(E, device=dev)[None]) | self.boundary  # the pair's left point
        self.bc = None if bc is None else torch.as_tensor(np.repeat(bc, Ff, axis=0), device=dev)
        spts = np.stack([x[coord[:, d]] for d in range(D)], 1)
        c = t(corners)
        self.pos = torch.einsum("sv,evd->sed", t(self._shape(spts)), c).cpu().numpy()
        self.G, self.det = self._metric(spts, c)
        G, _ = self._metric(np.array(ref), c)
        n = torch.einsum("fr,rfex->fex", self.tn, G)
        self.dA = n.norm(dim=2)
        self.n = n / self.dA[..., None]
        self.volume = torch.einsum("s,se->e", self.w, self.det)

    def _signs(self):
        q = [(-1, -1), (1, -1), (1, 1), (-1, 1)]
        return np.array(q if self.D == 2 else [(*v, -1) for v in q] + [(*v, 1) for v in q], dtype=float)

    def _shape(self, p):
        return np.prod(0.5 * (1.0 + p[:, None] * self._signs()[None]), axis=2)

    def _metric(self, p, corners):
        """[r][pt][e][x] det * d xi_r / d x, and det."""
        sg, D = self._signs(), self.D
        f = 0.5 * (1.0 + p[:, None] * sg[None])
        J = []
        for r in range(D):
            h = f.copy()
            h[:, :, r] = 0.5 * sg[None, :, r]
            J.append(torch.einsum("sv,evd->sed", torch.as_tensor(h.prod(2), device=corners.device), corners))
        if D == 2:
            G = torch.stack([torch.stack([J[1][..., 1], -J[1][..., 0]], -1),
                             torch.stack([-J[0][..., 1], J[0][..., 0]], -1)])
        else:
            G = torch.stack([torch.linalg.cross(J[1], J[2]), torch.linalg.cross(J[2], J[0]),
                             torch.linalg.cross(J[0], J[1])])
        return G, (J[0] * G[0]).sum(-1)

    def apply(self, A, U):
        return (A @ U.reshape(U.shape[0], -1)).reshape((A.shape[0],) + U.shape[1:])

    def pressure(self, U):
        return (GAMMA - 1.0) * (U[..., -1] - 0.5 * (U[..., 1:-1] ** 2).sum(-1) / U[..., 0])

    def flux(self, U):
        """Inviscid flux, a list over the directions."""
        p, D = self.pressure(U), self.D
        out = []
        for d in range(D):
            v = U[..., d + 1] / U[..., 0]
            F = U * v[..., None]
            F[..., d + 1] += p
            F[..., -1] += p * v
            out.append(F)
        return out

    def viscous_flux(self, U, g):
        """Viscous flux from the conservative gradient g[d]; in 3-D with the stresses as the reference
        scheme writes them (tau_xz = mu (u_z + v_x), tau_yz = mu (u_z + v_y), the x flux of rho w
        -tau_zz)."""
        D, mu = self.D, 1.0 / TGV_RE
        rho, v = U[..., 0], [U[..., d + 1] / U[..., 0] for d in range(self.D)]
        dv = [[(g[x][..., i + 1] - g[x][..., 0] * v[i]) / rho for i in range(D)] for x in range(D)]
        e = U[..., -1] / rho - 0.5 * sum(a * a for a in v)
        de = []
        for x in range(D):
            dk = 0.5 * sum(a * a for a in v) * g[x][..., 0] + rho * sum(a * b for a, b in zip(v, dv[x]))
            de.append((g[x][..., -1] - dk - g[x][..., 0] * e) / rho)
        div = sum(dv[d][d] for d in range(D)) / 3.0
        k = mu * GAMMA / TGV_PR
        diag = [2.0 * mu * (dv[d][d] - div) for d in range(D)]
        xy = mu * (dv[1][0] + dv[0][1])
        xz, yz = mu * (dv[2][0] + dv[0][1]), mu * (dv[2][0] + dv[1][1])
        tau = [[diag[0], xy, xz], [xy, diag[1], yz], [xz, yz, diag[2]]]
        rows = [[diag[0], xy, diag[2]], tau[1], tau[2]]
        out = []
        for d in range(D):
            heat = sum(v[i] * tau[d][i] for i in range(D)) + k * de[d]
            out.append(-torch.stack([torch.zeros_like(rho)] + rows[d] + [heat], -1))
        return out

    def speeds(self, Uf):
        vn = (Uf[..., 1:-1] * self.n).sum(-1) / Uf[..., 0]
        return vn.abs() + torch.sqrt(torch.clamp(GAMMA * self.pressure(Uf) / Uf[..., 0], min=0.0))

    def outside(self, Uf, free):
        """The state across every flux point."""
        UR = Uf.reshape(-1, Uf.shape[-1])[self.across.reshape(-1)].reshape(Uf.shape)
        if self.bc is None:
            return UR
        rho, vel, p = Uf[..., 0], Uf[..., 1:-1] / Uf[..., :1], self.pressure(Uf)
        n = self.n
        vn = (vel * n).sum(-1)
        wall = torch.cat([Uf[..., :1], rho[..., None] * (vel - 2.0 * vn[..., None] * n), Uf[..., -1:]], -1)
        rb, vb, pb = free
        vB = torch.zeros_like(vel)
        vB[..., 0] = vb
        gm = GAMMA - 1.0
        vnB = (vB * n).sum(-1)
        cL, cB = torch.sqrt(GAMMA * p / rho), math.sqrt(GAMMA * pb / rb)
        fast = vnB.abs() >= cB
        RL = torch.where(fast & (vn >= 0), vnB + 2.0 / gm * cB, vn + 2.0 / gm * cL)
        RB = torch.where(fast & (vn < 0), vn - 2.0 / gm * cL, vnB - 2.0 / gm * cB)
        c = 0.25 * gm * (RL - RB)
        s = torch.where(vn < 0, torch.full_like(p, rb ** GAMMA / pb), rho ** GAMMA / p)
        rR = (c * c / GAMMA * s) ** (1.0 / gm)
        pR = c * c * rR / GAMMA
        V = 0.5 * (RL + RB)
        vR = torch.where((vn < 0)[..., None], vB + (V - vnB)[..., None] * n, vel + (V - vn)[..., None] * n)
        far = torch.cat([rR[..., None], rR[..., None] * vR, (pR / gm + 0.5 * rR * (vR * vR).sum(-1))[..., None]], -1)
        UR = torch.where((self.boundary & (self.bc == 8))[..., None], wall, UR)
        return torch.where((self.boundary & (self.bc == 1))[..., None], far, UR)

    def normal(self, F):
        return sum(self.n[..., d:d + 1] * F[d] for d in range(self.D))

    def roe(self, UL, UR):
        n, g = self.n, GAMMA
        vL, vR = UL[..., 1:-1] / UL[..., :1], UR[..., 1:-1] / UR[..., :1]
        pL, pR = self.pressure(UL), self.pressure(UR)
        hL, hR = (UL[..., -1] + pL) / UL[..., 0], (UR[..., -1] + pR) / UR[..., 0]
        sq = torch.sqrt(UR[..., 0] / UL[..., 0])
        r = 1.0 / (sq + 1.0)
        um = r[..., None] * (vL + sq[..., None] * vR)
        hm = r * (hL + sq * hR)
        usq, unm = 0.5 * (um * um).sum(-1), (um * n).sum(-1)
        a2 = (g - 1.0) * (hm - usq)
        a = torch.sqrt(a2)
        vnL, vnR = (vL * n).sum(-1), (vR * n).sum(-1)
        eps = 0.5 * ((vnL - vnR).abs() + (torch.sqrt(g * pL / UL[..., 0]) - torch.sqrt(g * pR / UR[..., 0])).abs())
        lam = []
        for v in (unm, unm + a, unm - a):
            v = v.abs()
            lam.append(torch.where(v < 2 * eps, 0.25 * v * v / torch.where(eps > 0, eps, torch.ones_like(eps)) + eps, v))
        l0, lp, lm = lam
        du = UR - UL
        b2, b3 = 0.5 * (lp + lm) - l0, 0.5 * (lp - lm) / a
        s = usq * du[..., 0] - (um * du[..., 1:-1]).sum(-1) + du[..., -1]
        t = unm * du[..., 0] - (n * du[..., 1:-1]).sum(-1)
        A, B = b2 * (g - 1.0) / a2 * s - b3 * t, b3 * (g - 1.0) * s - b2 * t
        diss = l0[..., None] * du
        diss = diss + torch.cat([A[..., None], A[..., None] * um + B[..., None] * n, (A * hm + B * unm)[..., None]], -1)
        return 0.5 * (self.normal(self.flux(UL)) + self.normal(self.flux(UR)) - diss)

    def residual(self, U, speed, free=None):
        """divF at the solution points; the wave speeds of each pair's left point are stored."""
        D = self.D
        Uf = self.apply(self.to_f, U)
        UR = self.outside(Uf, free)
        lam = torch.maximum(self.speeds(Uf), self.speeds(UR))
        common = 0.5 * (self.normal(self.flux(Uf)) + self.normal(self.flux(UR)) - lam[..., None] * (UR - Uf))
        if self.riemann:
            common = self.roe(Uf, UR)
        else:
            speed.copy_(torch.where(self.first, lam, speed))
        F = self.flux(U)
        if self.viscous:
            jump = 0.5 * (UR - Uf)
            ref = [self.apply(self.grad[d], U) + self.apply(self.corr * self.tn[:, d][None], jump) for d in range(D)]
            g = [sum(self.G[r][..., x:x + 1] * ref[r] for r in range(D)) / self.det[..., None] for x in range(D)]
            F = [a + b for a, b in zip(F, self.viscous_flux(U, g))]
            own = self.normal(self.viscous_flux(Uf, [self.apply(self.to_f, a) for a in g]))
            # the neighbour's flux along this side's normal is the negative of its own
            other = own.reshape(-1, own.shape[-1])[self.across.reshape(-1)].reshape(own.shape)
            common = common + 0.5 * (own - other) + (Uf - UR)
        T = [sum(self.G[r][..., x:x + 1] * F[x] for x in range(D)) for r in range(D)]
        inner = sum(self.apply(self.to_f * self.tn[:, r:r + 1], T[r]) for r in range(D))
        div = sum(self.apply(self.grad[r], T[r]) for r in range(D))
        return div + self.apply(self.corr, common * self.dA[..., None] - inner)

    def element_dt(self, speed, cfl):
        around = torch.einsum("fe,f,fe->e", speed, self.w_face, self.dA)
        return cfl * CFL_LIMIT[self.P] * 2.0 * self.volume / around


def _box_mesh(case):
    """Corners and neighbours of a periodic box, elements numbered [z][x][y]."""
    D, n, lo, side = _box(case)
    h = side / n
    grid = np.stack(np.meshgrid(*[lo + h * np.arange(n + 1)] * D, indexing="ij"), -1)
    if case["kind"] == "vortex2d":
        i, j = np.meshgrid(np.arange(n + 1), np.arange(n + 1), indexing="ij")
        inner = (i > 0) & (i < n) & (j > 0) & (j < n)
        grid = grid + np.where(inner[..., None], _jitter(j * (n + 1) + i, 0.1 * np.array([h, h])), 0.0)
    return _structured(grid, (n,) * D, periodic=True)


def _jitter(vertex, amp):
    """Displacement of a vertex: splitmix64 of the mesh seed and the vertex' coordinate number."""
    out = []
    for d, a in enumerate(amp):
        x = (np.uint64(MESH_SEED) ^ (vertex * 2 + d).astype(np.uint64)) + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        x = x ^ (x >> np.uint64(31))
        out.append((2.0 * (x >> np.uint64(11)).astype(np.float64) / 9007199254740992.0 - 1.0) * a)
    return np.stack(out, -1)


def _channel_mesh(nx, ny):
    xs = np.linspace(-1.5, 1.5, nx + 1)
    yb = 0.0625 * np.exp(-25.0 * xs * xs)
    i, j = np.meshgrid(np.arange(nx + 1), np.arange(ny + 1), indexing="ij")
    grid = np.stack([xs[i], yb[i] + (0.8 - yb[i]) * (j / ny)], -1)
    inner = (i > 0) & (i < nx) & (j > 0) & (j < ny)
    grid = grid + np.where(inner[..., None], _jitter(j * (nx + 1) + i, 0.1 * np.array([3.0 / nx, 0.8 / ny])), 0.0)
    return _structured(grid, (nx, ny), periodic=False)


def _structured(grid, n, periodic):
    """(corners [E][2^D][D], neighbours [2D][E], boundary numbers) of a logically Cartesian grid."""
    D = len(n)
    q = [(0, 0), (1, 0), (1, 1), (0, 1)]
    offsets = q if D == 2 else [(*v, 0) for v in q] + [(*v, 1) for v in q]
    idx = np.stack(np.meshgrid(*[np.arange(m) for m in n], indexing="ij"), -1)
    order = (0, 1) if D == 2 else (2, 0, 1)  # slowest index first
    cell = idx.transpose(order + (D,)).reshape(-1, D)
    number = np.zeros(n, dtype=np.int64)
    number[tuple(cell.T)] = np.arange(len(cell))
    corners = np.stack([grid[tuple((cell + np.array(o)).T)] for o in offsets], 1)
    nb, bc = [], []
    for dim, side, _ in _FACES[D]:
        to = cell.copy()
        to[:, dim] += side
        out = (to[:, dim] < 0) | (to[:, dim] >= n[dim])
        to[:, dim] %= n[dim]
        nb.append(np.where(out & (not periodic), -1, number[tuple(to.T)]))
        bc.append(np.full(len(cell), 1 if dim == 0 else 8))
    return corners, np.array(nb), None if periodic else np.array(bc)


class _Level:
    """A scheme with its state: the RK update of one context."""

    def __init__(self, scheme, U, time_type, cfl=None, dt=None, local=False, free=None, a=None):
        self.s, self.time_type, self.cfl, self.dt, self.local, self.free, self.a = scheme, time_type, cfl, dt, local, free, a
        self.U = torch.as_tensor(U, dtype=torch.float64, device=_device())
        self.refresh()

    def refresh(self):
        self.speed = self.s.speeds(self.s.apply(self.s.to_f, self.U))

    def residual(self):
        return self.s.residual(self.U, self.speed, self.free)

    def update(self, first=False, src=None):
        """One step; returns the residual of its first stage."""
        if first:
            self.refresh()
        dt = self.dt
        if self.cfl is not None:
            dt = self.s.element_dt(self.speed, self.cfl)
            self.dt_used = dt = dt[None, :, None] if self.local else dt.min()
        U0, total, kept = self.U, 0.0, None
        det = self.s.det[..., None]
        a, b = (self.a, None) if self.time_type == 6 else ([0.5, 0.5, 1.0], [1 / 6, 1 / 3, 1 / 3, 1 / 6])
        for k in range(4):
            r = self.residual()
            kept = r if k == 0 else kept
            r = r if src is None else r + src
            if b is not None:
                total = total + b[k] * r
            if b is None or k < 3:
                self.U = U0 - a[k] * r / det * dt
        if b is not None:
            self.U = U0 - total / det * dt
            self.last = r
        return kept


def _cycle(levels, restrict, prolong, smooth):
    """One P-multigrid V-cycle (full approximation scheme) over levels of ascending order."""
    top = len(levels) - 1
    U, r, sources, starts = levels[top].U, levels[top].residual(), [None] * top, [None] * top
    for i in range(top - 1, -1, -1):
        g = levels[i]
        g.U = g.s.apply(restrict[i], U)
        sources[i] = g.s.apply(restrict[i], r) - g.residual()
        starts[i] = g.U
        for _ in range(smooth):
            g.update(src=sources[i])
        if i > 0:
            U, r = g.U, g.residual() + sources[i]
    for i in range(top):
        g = levels[i]
        for _ in range(smooth):
            g.update(src=sources[i])
        levels[i + 1].U = levels[i + 1].U + g.s.apply(prolong[i], g.U - starts[i])


def _tensor(a, D):
    """The D-fold tensor product of a 1-D operator, first dimension fastest."""
    out = a
    for _ in range(D - 1):
        out = np.kron(a, out)
    return torch.as_tensor(out, dtype=torch.float64, device=_device())


def _channel_step(nx, ny, order, mach, seed):
    """A channel's state after one update and one cycle."""
    corners, nb, bc = _channel_mesh(nx, ny)
    free = (1.0, mach, 1.0 / GAMMA)
    a = [0.153, 0.442, 0.931, 1.0] if order <= 2 else [0.158, 0.477, 1.0, 1.0]
    levels = []
    for q in range(order + 1):
        s = _Scheme(2, q, corners, nb, bc)
        U = _channel_state(s.pos, mach, seed)
        if q < order:  # a coarse level starts from the free stream
            U[...] = [1.0, mach, 0.0, 1.0 / GAMMA / (GAMMA - 1.0) + 0.5 * mach * mach]
        levels.append(_Level(s, U, 6, cfl=0.9, local=True, free=free, a=a))
    x = [lv.s.points for lv in levels]
    levels[-1].update(first=True)
    _cycle(levels, [_tensor(_lagrange(x[q + 1], x[q]), 2) for q in range(order)],
           [_tensor(_lagrange(x[q], x[q + 1]), 2) for q in range(order)], 2)
    return levels[-1].U


def exact(case, seed):
    if case["do"] == "batch":
        parts = {}
        for i, (nx, ny, order, mach) in enumerate(_channels(case)):
            parts.setdefault("P%d" % order, []).append(_channel_step(nx, ny, order, mach, seed * 1000 + i))
        return {k: torch.cat(v, 1) for k, v in parts.items()}
    if case["do"] == "pmg":
        return {"U": _channel_step(case["nx"], case["ny"], case["order"], case["mach"], seed)}
    corners, nb, _ = _box_mesh(case)
    D = corners.shape[2]
    scheme = _Scheme(D, case["order"], corners, nb, None, bool(case.get("viscous")), case.get("riemann", 0))
    U = _initial(case, scheme.pos, seed)
    if case["kind"] == "tgv3d":
        level = _Level(scheme, U, 4, dt=_tgv_dt(case))
    else:
        level = _Level(scheme, U, 4, cfl=0.5)
    for k in range(case.get("steps", 1)):
        r0 = level.update(first=k == 0)
    out = {"U": level.U}
    if case["do"] == "monitor":
        out["dt"] = level.dt
        out["residual"] = torch.sqrt(torch.einsum("sek,se,s->k", r0 * r0, 1.0 / scheme.det, scheme.w)).cpu().numpy()
    if case["do"] == "members":
        out["divF"] = level.last
    return out
