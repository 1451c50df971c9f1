"""Timed workloads of the LW-FR / MDRK library, through its public entry points.

Each case is a mesh, a scheme and one call a user's program makes: a right-hand
side (``rhs``), a run of the device-resident ``solve_lwfr`` loop (``solve_lwfr``
itself, or the C ABI's set_state_dev / solve_init / advance / get_state_dev on
states that live on the GPU), an ensemble's steps, or a checkpointed gradient.
``exact`` evaluates the same scheme in plain torch float64 without the library.
"""
from __future__ import annotations

import ctypes as C
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "trixilw.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import trixilw_hip as tlw  # noqa: E402
from trixilw_hip import _lib  # noqa: E402

GAMMA = 1.4
MU, PR = 0.01, 0.72


# --------------------------------------------------------------------------- cases
def listed():
    return [
        # one rhs! call on a small mesh: a host code with its own time loop; launches and latency
        dict(name="rhs_n3_16", kind="rhs", mesh="tree", level=4, order="morton", N=3, td="lw", phys="euler"),
        # the 32² vortex solved to t = 1 by solve_lwfr: a whole small run, from the initial state to the solution
        dict(name="solve_n4_32", kind="solve", mesh="tree", level=5, order="lexicographic", N=4, td="lw",
             phys="euler", t_final=1.0, steps=0),
        # the benchmark's 1024² vortex mesh, device-resident steps: a large production run
        dict(name="loop_n4_1024", kind="loop", mesh="tree", level=10, order="strips", N=4, td="lw", phys="euler",
             steps=10),
        # polydeg 3 in Trixi's tree order (the mesh's default)
        dict(name="loop_n3_512", kind="loop", mesh="tree", level=9, order="morton", N=3, td="lw", phys="euler",
             steps=10),
        # the two-stage MDRK scheme, two right-hand sides a step
        dict(name="loop_mdrk_n3_512", kind="loop", mesh="tree", level=9, order="strips", N=3, td="mdrk",
             phys="euler", steps=6),
        # compressible Navier-Stokes on the TreeMesh (BR1 gradients in every Taylor level)
        dict(name="loop_ns_n4_256", kind="loop", mesh="tree", level=8, order="strips", N=4, td="lw", phys="ns",
             steps=6),
        # a warped StructuredMesh of ragged size in Trixi's linear order
        dict(name="loop_curved_n4_301x217", kind="loop", mesh="curved", nx=301, ny=217, order="lexicographic", N=4,
             td="lw", phys="euler", steps=8),
        # curvilinear Navier-Stokes with MDRK at 128²: many short steps, replayed from a captured graph
        dict(name="loop_curved_ns_mdrk_n3_128", kind="loop", mesh="curved", nx=128, ny=128, order="strips", N=3,
             td="mdrk", phys="ns", steps=20, graphs=True),
        # a four-quadrant Riemann problem: shock-capturing blend, time-averaged Dirichlet boundaries
        dict(name="loop_riemann_sc_n4_256", kind="loop", mesh="tree", level=8, order="strips", N=4, td="lw",
             phys="sc", steps=8),
        # a TreeMesh whose centre is refined once: L2 mortars between levels
        dict(name="loop_refined_n4_128", kind="loop", mesh="refined", level=7, box=0.5, N=4, td="lw", phys="euler",
             steps=8),
        # 64 instances of both polynomial degrees, 16² to 128² elements, in one launch per kernel and step
        dict(name="ensemble_64", kind="ensemble", instances=64, draw=2024, steps=10),
        # gradient of the kinetic energy after 40 steps with respect to the initial state
        dict(name="gradient_n4_64", kind="gradient", mesh="tree", level=6, order="lexicographic", N=4, td="lw",
             phys="euler", steps=40, every=20),
    ]


def draw(rng):
    """One more case of the same ranges: every kind of call, sizes spread over their logarithm, odd ones too."""
    pick = rng.choice(["rhs", "solve", "loop", "loop", "mdrk", "ns", "curved", "curved", "curved_ns", "sc",
                       "refined", "ensemble", "gradient"])
    N = rng.choice([3, 4])
    order = rng.choice(["morton", "strips", "lexicographic"])
    tree = dict(mesh="tree", order=order, N=N, td="lw", phys="euler")

    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if pick == "rhs":
        if rng.random() < 0.5:
            return dict(kind="rhs", mesh="curved", nx=side(5, 400), ny=side(5, 400), order="lexicographic", N=N,
                        td="lw", phys="euler")
        return dict(tree, kind="rhs", level=rng.randint(3, 9))
    if pick == "solve":
        return dict(tree, kind="solve", level=rng.randint(4, 7), t_final=0.0, steps=rng.randint(10, 70))
    if pick == "loop":
        return dict(tree, kind="loop", level=rng.randint(5, 9), steps=rng.randint(4, 15))
    if pick == "mdrk":
        return dict(tree, kind="loop", level=rng.randint(5, 9), td="mdrk", steps=rng.randint(3, 8))
    if pick == "ns":
        return dict(tree, kind="loop", level=rng.randint(4, 8), phys="ns", td=rng.choice(["lw", "mdrk"]),
                    steps=rng.randint(3, 8))
    if pick in ("curved", "curved_ns"):
        return dict(kind="loop", mesh="curved", nx=side(17, 320), ny=side(17, 320),
                    order=rng.choice(["lexicographic", "strips"]), N=N, td=rng.choice(["lw", "mdrk"]),
                    phys="euler" if pick == "curved" else "ns", steps=rng.randint(3, 10))
    if pick == "sc":
        return dict(tree, kind="loop", level=rng.randint(5, 8), phys="sc", steps=rng.randint(3, 10))
    if pick == "refined":
        return dict(kind="loop", mesh="refined", level=rng.randint(4, 7), box=rng.choice([0.25, 0.5, 0.75]), N=N,
                    td=rng.choice(["lw", "mdrk"]), phys="euler", steps=rng.randint(4, 10))
    if pick == "ensemble":
        return dict(kind="ensemble", instances=rng.randint(9, 64), draw=rng.randint(1, 10000),
                    steps=rng.randint(4, 12))
    return dict(tree, kind="gradient", level=rng.randint(4, 6), td=rng.choice(["lw", "mdrk"]),
                steps=rng.randint(5, 40), every=rng.randint(3, 20))


# --------------------------------------------------------------------------- inputs
def _dev():
    return torch.device("cuda")


def _params(seed, n):
    g = torch.Generator().manual_seed(int(seed) * 7919 + 17)
    return [float(v) for v in torch.rand(n, generator=g, dtype=torch.float64)]


def _pack(rho, v1, v2, p):
    return torch.stack([rho, rho * v1, rho * v2, p / (GAMMA - 1.0) + 0.5 * rho * (v1 * v1 + v2 * v2)], dim=-1)


def _vortex(x, y, L, strength, mach, seed):
    """Isentropic vortex in a periodic box of side L with a smooth density perturbation of one per cent."""
    r = _params(seed, 8)
    cx, cy = L * (0.3 * r[0] - 0.15), L * (0.3 * r[1] - 0.15)
    dx, dy = x - cx, y - cy
    dx = dx - L * torch.floor(dx / L + 0.5)
    dy = dy - L * torch.floor(dy / L + 0.5)
    s = 20.0 / L
    dx, dy = s * dx, s * dy
    r2 = dx * dx + dy * dy
    a = strength / (2.0 * math.pi) * torch.exp(0.5 * (1.0 - r2))
    T = 1.0 - (GAMMA - 1.0) * strength**2 / (8.0 * GAMMA * math.pi**2) * torch.exp(1.0 - r2)
    w = 2.0 * math.pi / L
    pert = 1.0 + 0.01 * (torch.sin(w * x + 6.0 * r[2]) * torch.cos(2.0 * w * y + 6.0 * r[3])
                         + torch.sin(3.0 * w * x + 6.0 * r[4]) * torch.sin(w * y + 6.0 * r[5]))
    v = mach * math.sqrt(GAMMA) / math.sqrt(2.0)
    rho = T ** (1.0 / (GAMMA - 1.0))
    return _pack(rho * pert, v - a * dy, v + a * dx, rho * T)


def _shear(x, y, L, seed):
    """Shear flow with density and pressure waves on a periodic box of side L."""
    r = _params(seed, 6)
    w = 2.0 * math.pi / L
    rho = 1.0 + 0.2 * torch.sin(w * x + 6.0 * r[0]) * torch.cos(w * y + 6.0 * r[1])
    v1 = 0.3 + 0.1 * torch.sin(w * y + 6.0 * r[2])
    v2 = -0.2 + 0.1 * torch.cos(w * x + 6.0 * r[3])
    p = 1.0 + 0.1 * torch.cos(w * (x + y) + 6.0 * r[4])
    return _pack(rho, v1, v2, p)


# Lax-Liu configuration 3 (ρ, v1, v2, p) in the quadrants NE, NW, SW, SE, split at 0.5
_QUAD = ((1.5, 0.0, 0.0, 1.5), (0.5323, 1.206, 0.0, 0.3), (0.138, 1.206, 1.206, 0.029), (0.5323, 0.0, 1.206, 0.3))


def _riemann(x, y, seed):
    """The quadrant data with a smooth density modulation of two per cent inside the domain."""
    r = _params(seed, 2)
    q = [torch.zeros_like(x) for _ in range(4)]
    east, north = x >= 0.5, y >= 0.5
    for k, m in enumerate((east & north, ~east & north, ~east & ~north, east & ~north)):
        for v in range(4):
            q[v] = torch.where(m, torch.full_like(x, _QUAD[k][v]), q[v])
    bump = torch.sin(math.pi * x) ** 2 * torch.sin(math.pi * y) ** 2
    rho = q[0] * (1.0 + 0.02 * bump * torch.cos(6.0 * x + 6.0 * r[0]) * torch.cos(6.0 * y + 6.0 * r[1]))
    return _pack(rho, q[1], q[2], q[3])


def _box(case):
    if case["phys"] == "sc":
        return 0.0, 1.0
    if case["mesh"] == "curved":
        return 0.0, 2.0 if case["phys"] == "ns" else 20.0
    return (-1.0, 1.0) if case["phys"] == "ns" else (-10.0, 10.0)


def _warp(lo, hi):
    L = hi - lo

    def mapping(xi, eta):
        s, t = 0.5 * (xi + 1.0), 0.5 * (eta + 1.0)
        w = 0.05 * np.sin(2.0 * np.pi * s) * np.sin(2.0 * np.pi * t)
        return lo + L * (s + w), lo + L * (t + w)

    return mapping


def _mesh(case):
    lo, hi = _box(case)
    if case["mesh"] == "curved":
        return tlw.StructuredMesh((case["nx"], case["ny"]), _warp(lo, hi), ordering=case["order"])
    if case["mesh"] == "refined":
        b = case["box"] * hi
        patch = {"type": "box", "coordinates_min": (-b, -b), "coordinates_max": (b, b)}
        return tlw.TreeMesh((lo, lo), (hi, hi), case["level"], refinement_patches=(patch,))
    return tlw.TreeMesh((lo, lo), (hi, hi), case["level"], periodicity=case["phys"] != "sc", ordering=case["order"])


def _coords(mesh, nodes):
    if getattr(mesh, "curved", False):
        x, y = mesh.node_coordinates(nodes)
        return torch.tensor(x, device=_dev()), torch.tensor(y, device=_dev())
    c = torch.from_numpy(np.ascontiguousarray(mesh.element_center)).to(_dev())
    h = 0.5 * torch.from_numpy(np.ascontiguousarray(mesh.element_length)).to(_dev())
    t = torch.from_numpy(np.ascontiguousarray(nodes)).to(_dev())
    x = c[:, 0, None, None] + h[:, None, None] * t[None, None, :]
    y = c[:, 1, None, None] + h[:, None, None] * t[None, :, None]
    n = len(nodes)
    return x.expand(-1, n, n), y.expand(-1, n, n)


def _initial(case, mesh, nodes, seed):
    x, y = _coords(mesh, nodes)
    lo, hi = _box(case)
    if case["phys"] == "sc":
        return _riemann(x, y, seed).contiguous()
    if case["phys"] == "ns":
        return _shear(x, y, hi - lo, seed).contiguous()
    r = _params(seed + 101, 2)
    mid = 0.5 * (lo + hi)
    return _vortex(x - mid, y - mid, hi - lo, 3.0 + 2.0 * r[0], 0.3 + 0.4 * r[1], seed).contiguous()


def _cfl(case):
    if case["phys"] == "sc":
        return 0.3
    if case["phys"] == "ns":
        return 0.5
    N = case["N"]
    return 0.98 * (N + 1) * (1.0, 0.333, 0.170, 0.103)[N - 1] * (0.5 if case["td"] == "mdrk" else 1.0)


def _semi(case, mesh):
    eq = tlw.CompressibleEulerEquations2D(GAMMA)
    td = tlw.MDRK() if case["td"] == "mdrk" else tlw.LW()
    vi, bc = tlw.VolumeIntegralFR(td), None
    if case["phys"] == "sc":
        bc = tlw.FourQuadrantRiemann()
        vi = tlw.VolumeIntegralFRShockCapturing(tlw.IndicatorHennemannGassner(eq, None, alpha_max=0.5), vi)
    solver = tlw.DGSEM(case["N"], volume_integral=vi)
    if case["phys"] == "ns":
        par = tlw.CompressibleNavierStokesDiffusion2D(eq, mu=MU, Prandtl=PR,
                                                     gradient_variables=tlw.GradientVariablesConservative())
        return tlw.SemidiscretizationHyperbolicParabolic(mesh, td, (eq, par), None, solver)
    return tlw.SemidiscretizationHyperbolic(mesh, td, eq, None, solver, boundary_conditions=bc)


class _Given:
    """An initial condition whose nodal values are given (solve_lwfr evaluates it once)."""

    def __init__(self, u):
        self.u = u.cpu().numpy()

    def __call__(self, x, y, t):
        return self.u


def prepare(case, seed):
    if case["kind"] == "ensemble":
        return _prepare_ensemble(case, seed)
    mesh = _mesh(case)
    semi = _semi(case, mesh)
    u = _initial(case, mesh, semi.solver.basis.nodes, seed)
    st = dict(case=case, semi=semi, u=u, cfl=_cfl(case))
    if case["kind"] == "rhs":
        st["dt"] = st["cfl"] * semi.max_dt(u)
        semi.cache["dt"][0] = st["dt"]
        st["du"] = torch.empty_like(u)
    elif case["kind"] == "solve":
        semi.initial_condition = _Given(u)
        tf = case["t_final"] if case["t_final"] > 0 else 1e9
        st["lw_update"] = tlw.semidiscretize(semi, semi.time_discretization, (0.0, tf))
    elif case["kind"] == "loop":
        st["out"] = torch.empty_like(u)
        if case.get("graphs"):
            st["stream"] = torch.cuda.Stream()
            _lib.check(_lib.lib().tlw_enable_graphs(semi.handle, 1), semi.handle)
    torch.cuda.synchronize()
    return st


def _members(case, seed):
    """(levels, degrees, Mach numbers, strengths) of the ensemble's instances, both degrees present."""
    levels, degs, machs, strengths = tlw.draw_vortex_ensemble(case["instances"], case["draw"])
    degs = np.array(degs)
    degs[0], degs[1] = 3, 4
    r = np.array(_params(seed, 2 * case["instances"]))
    k = case["instances"]
    return levels, degs, machs * (0.9 + 0.2 * r[:k]), strengths * (0.9 + 0.1 * r[k:])


def _ensemble_states(case, seed, N, nodes, meshes):
    levels, degs, machs, strengths = _members(case, seed)
    parts = []
    for mesh, k in zip(meshes, np.nonzero(degs == N)[0]):
        x, y = _coords(mesh, nodes)
        parts.append(_vortex(x, y, 20.0, float(strengths[k]), float(machs[k]), seed * 64 + int(k)))
    return parts


def _ensemble_meshes(case, seed, N):
    levels, degs, _, _ = _members(case, seed)
    return [tlw.TreeMesh((-10.0, -10.0), (10.0, 10.0), int(levels[k]), ordering="morton")
            for k in np.nonzero(degs == N)[0]]


def _prepare_ensemble(case, seed):
    eq = tlw.CompressibleEulerEquations2D(GAMMA)
    batches, cfls, u0s = [], [], []
    for N in (3, 4):
        meshes = _ensemble_meshes(case, seed, N)
        solver = tlw.DGSEM(N)
        batches.append(tlw.SemidiscretizationBatch(meshes, tlw.LW(), eq, [None] * len(meshes), solver))
        cfls.append(tlw.trixi2lw(0.98, solver))
        u0s.append(torch.cat(_ensemble_states(case, seed, N, solver.basis.nodes, meshes)).contiguous())
    ens = tlw.SemidiscretizationEnsemble(batches)
    st = dict(case=case, ens=ens, batches=batches, cfls=cfls, u0s=u0s, stream=torch.cuda.Stream(),
              outs=[torch.empty_like(u) for u in u0s])
    L = _lib.lib()
    _lib.check(L.tlw_ensemble_set_stream(ens._h, C.c_void_p(st["stream"].cuda_stream)), None)
    _lib.check(L.tlw_ensemble_enable_graphs(ens._h, 1), None)
    torch.cuda.synchronize()
    return st


# --------------------------------------------------------------------------- one pass
def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _loop(st):
    """A run of the device loop on device-resident states, as a C ABI host drives it."""
    semi, L, h = st["semi"], _lib.lib(), st["semi"].handle
    semi._bind_stream()
    _lib.check(L.tlw_set_state_dev(h, _ptr(st["u"])), h)
    _lib.check(L.tlw_solve_init(h, 0.0, float("inf"), st["cfl"]), h)
    _lib.check(L.tlw_advance(h, st["case"]["steps"], None, None, None, None), h)
    _lib.check(L.tlw_get_state_dev(h, _ptr(st["out"])), h)
    return st["out"]


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "rhs":
        tlw.rhs(st["du"], st["u"], st["semi"], 0.0)
        return st["du"]
    if kind == "solve":
        sol = tlw.solve_lwfr(st["lw_update"], (), 1e-6, None, time_step_computation=tlw.CFLBased(st["cfl"]),
                             max_steps=case["steps"] or None)
        return [sol.u, sol.t]
    if kind == "loop":
        if "stream" not in st:
            return _loop(st)
        main, side = torch.cuda.current_stream(), st["stream"]
        side.wait_stream(main)
        with torch.cuda.stream(side):
            out = _loop(st)
        main.wait_stream(side)
        return out
    if kind == "ensemble":
        L, ens = _lib.lib(), st["ens"]
        main, side = torch.cuda.current_stream(), st["stream"]
        side.wait_stream(main)
        for b, u in zip(ens.batches, st["u0s"]):
            _lib.check(L.tlw_set_state_dev(b.handle, _ptr(u)), b.handle)
        _lib.check(L.tlw_ensemble_solve_init(ens._h, 0.0, float("inf"), st["cfls"][0], st["cfls"][1]), None)
        ens.advance(case["steps"])
        for b, o in zip(ens.batches, st["outs"]):
            _lib.check(L.tlw_get_state_dev(b.handle, _ptr(o)), b.handle)
        main.wait_stream(side)
        return st["outs"]
    J, grad, u, dts = tlw.gradient_lw(st["semi"], st["u"], case["steps"], st["cfl"],
                                      checkpoint_every=case["every"])
    return [J, grad, u]


# --------------------------------------------------------------------------- accounting
def _elements(case):
    if case["mesh"] == "curved":
        return case["nx"] * case["ny"]
    if case["mesh"] == "refined":  # the box's share of the cells is split in four
        side = 2 * int(round(case["box"] * 2 ** (case["level"] - 1)))
        return 4 ** case["level"] + 3 * side * side
    return 4 ** case["level"]


def _steps(case):
    if case["kind"] == "rhs":
        return 1
    if case["kind"] == "solve" and not case["steps"]:  # CFL steps to t_final at speeds of about 1.3 + 1.2
        h = 20.0 / 2 ** case["level"]
        return max(1, round(case["t_final"] * 5.0 / (_cfl(case) * h)))
    return case["steps"]


def _work_of(E, N, td, phys, curved, steps):
    """State in and out per stage (64 bytes a node, MDRK: 3 reads and 2 writes a step), the metric terms of a
    curvilinear mesh (40 bytes a node and stage), and the flops of the Taylor procedure: per stage the Euler
    (22) or Navier-Stokes (90) flux pairs, their 8-term stencils, and the derivative contractions."""
    n = N + 1
    dofs = E * n * n
    stages = 1 if td == "lw" else 2
    io = 64.0 if td == "lw" else 160.0
    if curved:
        io += 40.0 * stages
    if td == "lw":
        nflux, ncon = (17, 5) if N == 4 else (11, 4)
    else:
        nflux, ncon = 15, 5
    per = nflux * ((90 if phys == "ns" else 22) + 16) + ncon * 16 * n
    if phys == "ns":
        per += ncon * 16 * n
    return dofs * steps * io, float(dofs * steps * per)


def work(case):
    if case["kind"] == "ensemble":
        levels, degs, _, _ = _members(case, 0)
        b = f = 0.0
        for lev, N in zip(levels, degs):
            bb, ff = _work_of(4 ** int(lev), int(N), "lw", "euler", False, case["steps"])
            b, f = b + bb, f + ff
        return {"bytes": b, "flops": f}
    b, f = _work_of(_elements(case), case["N"], case["td"], case["phys"], case["mesh"] == "curved", _steps(case))
    if case["kind"] == "gradient":  # the forward run, its recomputation and a reverse sweep of twice the forward
        b, f = 3.0 * b, 4.0 * f
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Four times the distance between the library and plain torch float64 over these ranges: on a uniform tree a
    run of steps agrees to a few 1e-15; on a curvilinear mesh the metric terms differ in their last bits
    (1.3e-13); a right-hand side alone loses the digits that the cancellation in D F̃ costs at small cells."""
    if case["kind"] == "rhs":
        return {"rel": 2e-11}
    if case["kind"] != "ensemble" and case["mesh"] == "curved":
        return {"rel": 1e-12}
    return {"rel": 2e-14}


# --------------------------------------------------------------------------- plain torch reference
def _gll(N):
    """Gauss-Lobatto-Legendre nodes, weights and the derivative matrix."""
    c = np.polynomial.legendre.Legendre.basis(N)
    x = np.concatenate([[-1.0], np.sort(c.deriv().roots().real), [1.0]])
    w = 2.0 / (N * (N + 1) * c(x) ** 2)
    n = N + 1
    bw = np.array([1.0 / np.prod([x[j] - x[k] for k in range(n) if k != j]) for j in range(n)])
    D = np.zeros((n, n))
    for i in range(n):
        for j in range(n):
            if i != j:
                D[i, j] = bw[j] / bw[i] / (x[i] - x[j])
        D[i, i] = -D[i].sum()
    return x, w, D


def _euler(u):
    v1, v2 = u[..., 1] / u[..., 0], u[..., 2] / u[..., 0]
    p = (GAMMA - 1.0) * (u[..., 3] - 0.5 * (u[..., 1] * v1 + u[..., 2] * v2))
    f = torch.stack([u[..., 1], u[..., 1] * v1 + p, u[..., 1] * v2, (u[..., 3] + p) * v1], -1)
    g = torch.stack([u[..., 2], u[..., 2] * v1, u[..., 2] * v2 + p, (u[..., 3] + p) * v2], -1)
    return f, g


def _viscous(u, gx, gy):
    rho = u[..., 0]
    v1, v2 = u[..., 1] / rho, u[..., 2] / rho
    p = (GAMMA - 1.0) * (u[..., 3] - 0.5 * rho * (v1 * v1 + v2 * v2))
    kappa = GAMMA / ((GAMMA - 1.0) * PR)

    def prim(q):
        a, b = (q[..., 1] - q[..., 0] * v1) / rho, (q[..., 2] - q[..., 0] * v2) / rho
        pd = (GAMMA - 1.0) * (q[..., 3] - 0.5 * q[..., 0] * (v1 * v1 + v2 * v2) - rho * (v1 * a + v2 * b))
        return a, b, (pd - q[..., 0] * p / rho) / rho

    v1x, v2x, Tx = prim(gx)
    v1y, v2y, Ty = prim(gy)
    t11, t12, t22 = 4 / 3 * v1x - 2 / 3 * v2y, v1y + v2x, 4 / 3 * v2y - 2 / 3 * v1x
    z = torch.zeros_like(rho)
    return (MU * torch.stack([z, t11, t12, v1 * t11 + v2 * t12 + kappa * Tx], -1),
            MU * torch.stack([z, t12, t22, v1 * t12 + v2 * t22 + kappa * Ty], -1))


_STENCIL = {1: ((-1 / 12, 2), (2 / 3, 1), (-2 / 3, -1), (1 / 12, -2)), 2: ((1.0, 1), (-2.0, 0), (1.0, -1)),
            "2w": ((-1 / 12, 2), (4 / 3, 1), (-2.5, 0), (4 / 3, -1), (-1 / 12, -2)),
            3: ((0.5, 2), (-1.0, 1), (1.0, -1), (-0.5, -2)),
            4: ((0.5, 2), (-2.0, 1), (3.0, 0), (-2.0, -1), (0.5, -2))}


class _Ref:
    """The scheme on a conforming or 2:1 refined mesh of elements [e, j, i, variable] in plain torch."""

    def __init__(self, case, mesh):
        d = _dev()
        self.case, self.N, self.n = case, case["N"], case["N"] + 1
        x, w, D = _gll(self.N)
        self.nodes = x
        Dh = -np.diag(1.0 / w) @ D.T @ np.diag(w)
        self.x, self.w, self.D, self.Dh = (torch.from_numpy(np.ascontiguousarray(a)).to(d) for a in (x, w, D, Dh))
        self.nbr = torch.from_numpy(np.asarray(mesh.neighbors, dtype=np.int64)).to(d)
        self.mort = np.asarray(getattr(mesh, "mortars", np.zeros((0, 5))), dtype=np.int64)
        self.curved = bool(getattr(mesh, "curved", False))
        self.ns, self.sc = case["phys"] == "ns", case["phys"] == "sc"
        if self.curved:
            X, Y = (torch.tensor(a, device=d) for a in mesh.node_coordinates(x))
            xx, xe, yx, ye = self.dx(X[..., None])[..., 0], self.dy(X[..., None])[..., 0], \
                self.dx(Y[..., None])[..., 0], self.dy(Y[..., None])[..., 0]
            self.Ja = (ye, -xe, -yx, xx)
            self.J = (1.0 / (xx * ye - xe * yx))[..., None]
        else:
            invj = 2.0 / torch.from_numpy(np.asarray(mesh.element_length, dtype=np.float64)).to(d)
            self.J = invj[:, None, None, None].expand(-1, self.n, self.n, 1)
        if len(self.mort):
            self._mortar_setup()

    def dx(self, f, M=None):
        M = self.D if M is None else M
        return torch.stack([sum(M[i, k] * f[:, :, k] for k in range(self.n)) for i in range(self.n)], 2)

    def dy(self, f, M=None):
        M = self.D if M is None else M
        return torch.stack([sum(M[i, k] * f[:, k] for k in range(self.n)) for i in range(self.n)], 1)

    def div(self, f, g, M=None):
        if self.curved:
            a, b, c, e = (q[..., None] for q in self.Ja)
            f, g = a * f + b * g, c * f + e * g
        return self.dx(f, M) + self.dy(g, M)

    def cart(self, gx, gy):
        if not self.curved:
            return self.J * gx, self.J * gy
        a, b, c, e = (q[..., None] for q in self.Ja)
        return self.J * (a * gx + c * gy), self.J * (b * gx + e * gy)

    @staticmethod
    def side(q, f):
        return (q[:, :, 0], q[:, :, -1], q[:, 0], q[:, -1])[f]

    def add_faces(self, out, lifts):
        """out plus per-face node contributions (list of four [e, node, variable])."""
        out = out.clone()
        out[:, :, 0] += lifts[0]
        out[:, :, -1] += lifts[1]
        out[:, 0] += lifts[2]
        out[:, -1] += lifts[3]
        return out

    def br1(self, u):
        gx, gy = self.dx(u, self.Dh), self.dy(u, self.Dh)
        avg = [0.5 * (self.side(u, f) + self.side(u, f ^ 1)[self.nbr[:, f]]) for f in range(4)]
        z = torch.zeros_like(avg[0])
        s = (-1.0 / self.w[0], 1.0 / self.w[-1])
        return self.cart(self.add_faces(gx, [s[0] * avg[0], s[1] * avg[1], z, z]),
                         self.add_faces(gy, [z, z, s[0] * avg[2], s[1] * avg[3]]))

    def flux(self, q):
        f, g = _euler(q[0])
        if self.ns:
            fv, gv = _viscous(*q)
            f, g = f - fv, g - gv
        return f, g

    def level(self, u):
        """A Taylor level: the time derivative, with its element-local gradient for Navier-Stokes."""
        return (u,) + self.cart(self.dx(u), self.dy(u)) if self.ns else (u,)

    def base(self, u):
        return (u,) + self.br1(u) if self.ns else (u,)

    def diff(self, lev, k):
        """The k-th time difference of the flux at the Taylor states of the levels."""
        key = "2w" if k == 2 and self.N == 4 else k
        f = g = 0.0
        for c, s in _STENCIL[key]:
            q = tuple(sum((float(s) ** m / math.factorial(m)) * lev[m][a] for m in range(len(lev) if s else 1))
                      for a in range(len(lev[0])))
            ff, gg = self.flux(q)
            f, g = f + c * ff, g + c * gg
        return f, g

    def averages(self, u, dt, stage, us=None):
        """(Ũ, F̃, G̃) of an LW step (stage 0) or an MDRK stage."""
        lev = [self.base(u)]
        f, g = self.flux(lev[0])
        if stage == 0:
            U, F, G = u, f, g
            for k in range(1, self.N + 1):
                lev.append(self.level(-dt * self.J * self.div(f, g)))
                f, g = self.diff(lev, k)
                c = 1.0 / math.factorial(k + 1)
                U, F, G = U + c * lev[k][0], F + c * f, G + c * g
            return U, F, G
        lev.append(self.level(-dt * self.J * self.div(f, g)))
        ft, gt = self.diff(lev, 1)
        a, b = (0.5, 0.125) if stage == 1 else (1.0, 1.0 / 6.0)
        U, F, G = a * u + b * lev[1][0], a * f + b * ft, a * g + b * gt
        if stage == 2:
            ls = [self.base(us)]
            ls.append(self.level(-dt * self.J * self.div(*self.flux(ls[0]))))
            ft, gt = self.diff(ls, 1)
            U, F, G = U + ls[1][0] / 3.0, F + ft / 3.0, G + gt / 3.0
        return U, F, G

    def speeds(self, u, f, normal=None):
        v1, v2 = u[..., 1] / u[..., 0], u[..., 2] / u[..., 0]
        p = (GAMMA - 1.0) * (u[..., 3] - 0.5 * (u[..., 1] * v1 + u[..., 2] * v2))
        c = torch.sqrt(GAMMA * p / u[..., 0])
        if normal is None:
            return (v1 if f < 2 else v2).abs(), c
        return (v1 * normal[0] + v2 * normal[1]).abs(), c * torch.sqrt(normal[0] ** 2 + normal[1] ** 2)

    def numflux(self, f, ul, ur, Ul, Ur, Fl, Fr, normal=None):
        jl, jr, sl, sr = (Ul, Ur, ul, ur) if self.curved else (ul, ur, Ul, Ur)
        al, cl = self.speeds(sl, f, normal)
        ar, cr = self.speeds(sr, f, normal)
        lam = torch.maximum(al, ar) + torch.maximum(cl, cr)
        return 0.5 * (Fl + Fr) - 0.5 * lam[..., None] * (jr - jl)

    def rusanov(self, f, ul, ur):
        k = 0 if f < 2 else 1
        return self.numflux(f, ul, ur, ul, ur, _euler(ul)[k], _euler(ur)[k])

    def rhs(self, u, dt, stage=0, us=None):
        U, F, G = self.averages(u, dt, stage, us)
        vol = self.div(F, G, self.Dh)
        blend = None
        if self.sc:
            vol, blend = self.subcell(u, vol)
        lifts = [None] * 4
        for f in (1, 3):  # the + faces; the - faces take the same fluxes
            nb = self.nbr[:, f]
            ok = nb >= 0
            nn = nb.clamp(min=0)
            Fn = F if f == 1 else G
            normal = None
            if self.curved:
                pair = (self.Ja[0], self.Ja[1]) if f == 1 else (self.Ja[2], self.Ja[3])
                nrm = [q[:, :, 0] if f == 1 else q[:, 0] for q in pair]
                normal = [q[nn] for q in nrm]
                Fl = normal[0][..., None] * self.side(F, f) + normal[1][..., None] * self.side(G, f)
                Fr = normal[0][..., None] * self.side(F, f ^ 1)[nn] + normal[1][..., None] * self.side(G, f ^ 1)[nn]
            else:
                Fl, Fr = self.side(Fn, f), self.side(Fn, f ^ 1)[nn]
            Fs = self.numflux(f, self.side(u, f), self.side(u, f ^ 1)[nn], self.side(U, f), self.side(U, f ^ 1)[nn],
                              Fl, Fr, normal)
            if self.sc:
                Fs = self.blended(f, u, Fs, blend, nn, dt)
            minus = torch.zeros_like(Fs)
            minus[nn[ok]] = Fs[ok]
            lifts[f], lifts[f ^ 1] = torch.where(ok[:, None, None], Fs, torch.zeros_like(Fs)), minus
        if self.sc:
            for f in range(4):
                b = torch.nonzero(self.nbr[:, f] < 0)[:, 0]
                lifts[f][b] = self.boundary(f, b, u, U, F if f < 2 else G, stage)
        if len(self.mort):
            self.mortars(u, U, F, G, lifts)
        s = (-1.0 / self.w[0], 1.0 / self.w[-1])
        return -self.J * self.add_faces(vol, [s[f & 1] * lifts[f] for f in range(4)])

    # shock capturing: Hennemann-Gassner factor, first-order subcell FV, blended interface flux
    def subcell(self, u, vol):
        n = self.n
        V = np.stack([np.polynomial.legendre.Legendre.basis(m)(self.nodes) * math.sqrt(m + 0.5) for m in range(n)], 1)
        Vi = torch.from_numpy(np.linalg.inv(V)).to(u.device)
        ind = (GAMMA - 1.0) * (u[..., 0] * u[..., 3] - 0.5 * (u[..., 1] ** 2 + u[..., 2] ** 2))
        m2 = self.dy(self.dx(ind[..., None], Vi), Vi)[..., 0] ** 2
        tot, c1, c2 = (m2[:, :k, :k].sum((1, 2)) for k in (n, n - 1, n - 2))
        e = torch.maximum((tot - c1) / tot, torch.where(c1 != 0, (c1 - c2) / c1, torch.zeros_like(c1)))
        thr, par = 0.5 * 10.0 ** (-1.8 * n**0.25), math.log((1 - 1e-4) / 1e-4)
        al = 1.0 / (1.0 + torch.exp(-par / thr * (e - thr)))
        al = torch.where(al < 1e-3, torch.zeros_like(al), al)
        al = torch.where(al > 1 - 1e-3, torch.ones_like(al), al).clamp(max=0.5)
        sm = al.clone()
        for f in range(4):
            nb = self.nbr[:, f]
            sm = torch.where(nb >= 0, torch.maximum(sm, 0.5 * al[nb.clamp(min=0)]), sm)
        fx = torch.zeros((u.shape[0], n, n + 1, 4), dtype=u.dtype, device=u.device)
        gy = torch.zeros((u.shape[0], n + 1, n, 4), dtype=u.dtype, device=u.device)
        fx[:, :, 1:-1] = self.rusanov(1, u[:, :, :-1], u[:, :, 1:])
        gy[:, 1:-1] = self.rusanov(3, u[:, :-1], u[:, 1:])
        fv = (fx[:, :, 1:] - fx[:, :, :-1]) / self.w[:, None] + (gy[:, 1:] - gy[:, :-1]) / self.w[:, None, None]
        a = sm[:, None, None, None]
        low = (fx[:, :, 1], fx[:, :, -2], gy[:, 1], gy[:, -2])
        return torch.where(a.abs() <= 1e-12, vol, (1.0 - a) * vol + a * fv), (sm, low)

    def blended(self, f, u, Fs, blend, nn, dt):
        sm, low = blend
        ul, ur = self.side(u, f), self.side(u, f ^ 1)[nn]
        fn = self.rusanov(f, ul, ur)
        alp = (0.5 * (sm + sm[nn]))[:, None, None]
        Fb = (1.0 - alp) * Fs + alp * fn
        c = dt * self.J[0, 0, 0, 0] / (0.5 * self.w[0])
        ok = torch.ones_like(alp[..., 0], dtype=torch.bool).expand(-1, self.n)
        for s in (ul - c * (Fb - low[f]), ur - c * (low[f ^ 1][nn] - Fb)):
            p = s[..., 3] - 0.5 * (s[..., 1] ** 2 + s[..., 2] ** 2) / s[..., 0]
            ok = ok & (s[..., 0] > 0) & (p > 0)
        return torch.where(ok[..., None], Fb, fn)

    def boundary(self, f, b, u, U, Fn, stage):
        """Time-averaged Dirichlet data (steady quadrant states) against the face's own averages."""
        X, Y = self.mesh_xy[0][b], self.mesh_xy[1][b]
        x, y = self.side(X, f), self.side(Y, f)
        ub = _quad_state(x, y)
        fb = _euler(ub)[0 if f < 2 else 1]
        own = (self.side(u, f)[b], self.side(U, f)[b], self.side(Fn, f)[b])
        if f & 1:
            return self.numflux(f, own[0], ub, own[1], ub, own[2], fb)
        return self.numflux(f, ub, own[0], ub, own[1], fb, own[2])

    # L2 mortars: interpolate the large side to the halves, project the fluxes back
    def _mortar_setup(self):
        n = self.n
        x, w = np.polynomial.legendre.leggauss(n + 2)
        V = np.stack([np.polynomial.legendre.Legendre.basis(m)(self.nodes) * math.sqrt(m + 0.5) for m in range(n)], 1)

        def leg(t):
            return np.stack([np.polynomial.legendre.Legendre.basis(m)(t) * math.sqrt(m + 0.5) for m in range(n)], 1)

        Vi = np.linalg.inv(V)
        self.fwd, self.rev = [], []
        for sh in (-1.0, 1.0):
            self.fwd.append(torch.from_numpy(leg(0.5 * (self.nodes + sh)) @ Vi).to(_dev()))
            P = V @ (leg(0.5 * (x + sh)).T @ (0.5 * w[:, None] * (leg(x) @ Vi)))
            self.rev.append(torch.from_numpy(np.ascontiguousarray(P)).to(_dev()))

    def mortars(self, u, U, F, G, lifts):
        for ori in (1, 2):
            for big in (1, 2):
                sel = self.mort[(self.mort[:, 3] == ori) & (self.mort[:, 4] == big)]
                if not len(sel):
                    continue
                m = torch.from_numpy(sel[:, :3]).to(u.device)
                fl = (1 if big == 1 else 0) + 2 * (ori - 1)  # the large element's face; the small ones take fl ^ 1
                Fn = F if ori == 1 else G
                L = [self.side(q, fl)[m[:, 2]] for q in (u, U, Fn)]
                acc = 0.0
                for half in (0, 1):
                    S = [self.side(q, fl ^ 1)[m[:, half]] for q in (u, U, Fn)]
                    Lh = [torch.einsum("lk,ekv->elv", self.fwd[half], q) for q in L]
                    a, b = (Lh, S) if big == 1 else (S, Lh)
                    Fs = self.numflux(fl, a[0], b[0], a[1], b[1], a[2], b[2])
                    lifts[fl ^ 1][m[:, half]] = Fs
                    acc = acc + torch.einsum("lk,ekv->elv", self.rev[half], Fs)
                lifts[fl][m[:, 2]] = acc

    def max_dt(self, u):
        rho = u[..., 0]
        v1, v2 = u[..., 1] / rho, u[..., 2] / rho
        p = (GAMMA - 1.0) * (u[..., 3] - 0.5 * (u[..., 1] * v1 + u[..., 2] * v2))
        c = torch.sqrt(GAMMA * p / rho)
        l1, l2 = v1.abs() + c, v2.abs() + c
        J = self.J[..., 0]
        if self.curved:
            a, b, d, e = self.Ja
            l1, l2 = (a * l1 + b * l2).abs() * J, (d * l1 + e * l2).abs() * J
            m = float((l1.amax((1, 2)) + l2.amax((1, 2))).max())
        else:
            m = float((J[:, 0, 0] * (l1.amax((1, 2)) + l2.amax((1, 2)))).max())
        dt = 2.0 / (self.n * m)
        if self.ns:
            kappa = GAMMA / ((GAMMA - 1.0) * PR)
            s = J if self.curved else J * J
            lv = float((s * max(4.0 * MU / 3.0, MU * kappa / PR) / rho).max()) * 2.0 * (2 * self.N + 1)
            dt = min(dt, 1.0 / ((m + lv) * 2.0 * (2 * self.N + 1)))
        return dt

    def step(self, u, dt):
        if self.case["td"] == "mdrk":
            us = u + dt * self.rhs(u, dt, 1)
            return u + dt * self.rhs(u, dt, 2, us)
        return u + dt * self.rhs(u, dt)


def _quad_state(x, y):
    out = torch.zeros(x.shape + (4,), dtype=x.dtype, device=x.device)
    east, north = x >= 0.5, y >= 0.5
    for k, m in enumerate((east & north, ~east & north, ~east & ~north, east & ~north)):
        s = _pack(*(torch.full_like(x, v) for v in _QUAD[k]))
        out = torch.where(m[..., None], s, out)
    return out


def _reference(case, mesh):
    r = _Ref(case, mesh)
    if case["phys"] == "sc":
        r.mesh_xy = _coords(mesh, r.nodes)
    return r


def _run_exact(ref, u, cfl, steps, t_final=None):
    t, k = 0.0, 0
    while (steps and k < steps) or (not steps and t < t_final * (1.0 - 1e-12)):
        dt = cfl * ref.max_dt(u)
        if t_final is not None and t + dt > t_final:
            dt = t_final - t
        u = ref.step(u, dt)
        t, k = t + dt, k + 1
    return u, t


def exact(case, seed):
    if case["kind"] == "ensemble":
        outs = []
        for N, cfl in ((3, 0.98 * 4 * 0.170), (4, 0.98 * 5 * 0.103)):
            meshes = _ensemble_meshes(case, seed, N)
            sub = dict(N=N, td="lw", phys="euler")
            parts = []
            for m, u in zip(meshes, _ensemble_states(case, seed, N, _gll(N)[0], meshes)):
                parts.append(_run_exact(_Ref(sub, m), u.contiguous(), cfl, case["steps"])[0])
            outs.append(torch.cat(parts))
        return outs
    mesh = _mesh(case)
    ref = _reference(case, mesh)
    u = _initial(case, mesh, ref.nodes, seed)
    cfl = _cfl(case)
    if case["kind"] == "rhs":
        return ref.rhs(u, cfl * ref.max_dt(u))
    if case["kind"] == "solve":
        u, t = _run_exact(ref, u, cfl, case["steps"], case["t_final"] or None)
        return [u, t]
    if case["kind"] == "loop":
        return _run_exact(ref, u, cfl, case["steps"])[0]
    states, dts = [u], []
    for _ in range(case["steps"]):
        dts.append(cfl * ref.max_dt(states[-1]))
        states.append(ref.step(states[-1], dts[-1]))
    q = states[-1].clone().requires_grad_(True)
    area = ref.w[:, None] * ref.w[None, :] / ref.J[..., 0] ** 2
    J = (area * 0.5 * (q[..., 1] ** 2 + q[..., 2] ** 2) / q[..., 0]).sum()
    lam, = torch.autograd.grad(J, q)
    for k in range(case["steps"] - 1, -1, -1):
        q = states[k].clone().requires_grad_(True)
        lam, = torch.autograd.grad(ref.step(q, dts[k]), q, lam)
    return [float(J.detach()), lam, states[-1]]
