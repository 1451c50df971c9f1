"""The surface launch split at the domain boundary (from 4096 node-per-lane workgroups on, 5 elements
each for N=4, 8 for N=3, the workgroups with a boundary face run apart): every kernel pair that is
split, in steps of the device loop, whose dt and admissibility test take both launches.  State and
time against the CPU oracle (1e-12 relative; another order of the same sums), the split itself from
tlw_launch_info.  One element of higher pressure, at the boundary or inside, holds the largest speed,
so that the next dt follows from the one launch or the other.  Inputs are seeded."""
import numpy as np
import pytest

from gpu_helpers import assert_close, launch_info, setup, setup_curved, to_dev, to_lex, torch_mod
from test_gpu_curved_sc_parity import with_jump
from test_gpu_mortar_parity import setup_refined
from test_gpu_ns_wall_parity import perturbed, setup_walls

pytestmark = pytest.mark.gpu


def with_hot_element(u, e, f=1.5):
    """Density and pressure raised by f in element e, the pressure by f² there: c grows by sqrt(f)."""
    u = u.copy()
    v = u[e, ..., 1:3] / u[e, ..., 0:1]
    p = 0.4 * (u[e, ..., 3] - 0.5 * u[e, ..., 0] * (v**2).sum(-1))
    u[e, ..., 0] *= f
    u[e, ..., 1:3] *= f
    u[e, ..., 3] = f * f * p / 0.4 + 0.5 * u[e, ..., 0] * (v**2).sum(-1)
    return u


def run(semi, u_dev, K, tsc, tf=float("inf"), dt0=1e-6, tol=None):
    """The solution after K steps or at tf."""
    import trixilw_hip as tlw

    lw_update = tlw.semidiscretize(semi, semi.time_discretization, (0.0, tf))
    lw_update.u0.copy_(u_dev)
    return tlw.solve_lwfr(lw_update, (), dt0, tol, time_step_computation=tsc, max_steps=K)


def case(oracle_mod, kind, N, td="lw"):
    import trixilw_hip as tlw

    if kind == "tree_sc":
        ic = tlw.FourQuadrantRiemann()
        return setup(oracle_mod, N, 8, td=td, periodic=False, domain=(0.0, 1.0), bc=ic, ic=ic, amp=0.0, sc=True,
                     keep_aux=False)
    if kind == "tree":
        ic = tlw.IsentropicVortex(center=(0.7, -0.4), period=(1e9, 1e9))
        return setup(oracle_mod, N, 8, td=td, periodic=False, bc=ic, ic=ic, keep_aux=False, ordering="strips")
    nx, ny = (160, 128) if N == 4 else (256, 128)
    if kind == "curved":
        return setup_curved(oracle_mod, N, nx, ny, A=0.02, td=td, periodic=False)
    if kind == "curved_wall":
        return setup_curved(oracle_mod, N, nx, ny, A=0.02, td=td, periodic=False, boundary=tlw.slip_wall_approximate)
    if kind == "curved_sc":
        semi, o, u, mesh = setup_curved(oracle_mod, N, nx, ny, A=0.02, td=td, periodic=False, sc=True,
                                        alpha_smooth=False)
        return semi, o, with_jump(o, u), mesh
    if kind == "walls":
        semi, o, mesh = setup_walls(oracle_mod, N, 8, td=td)
        return semi, o, perturbed(o, 3, amp=1e-3), mesh
    box = ({"type": "box", "coordinates_min": (-6.0, -6.0), "coordinates_max": (6.0, 6.0)},)
    return setup_refined(oracle_mod, N, level=7, td=td, periodic=False, patches=box)


CASES = [("tree_sc", 4, "lw"), ("tree_sc", 3, "lw"), ("tree", 4, "lw"), ("tree", 3, "mdrk"), ("curved", 4, "lw"),
         ("curved", 3, "mdrk"), ("curved_wall", 4, "lw"), ("curved_sc", 4, "lw"), ("curved_sc", 3, "lw"),
         ("walls", 3, "lw"), ("walls", 4, "mdrk")]


# (the oracle's connectivity of the refined mesh takes ten seconds: once)
@pytest.mark.parametrize("kind,N,td,hot", [(*c, h) for c in CASES for h in ("corner", "inside")]
                         + [("refined", 4, "lw", "corner")])
def test_split_steps(oracle_mod, kind, N, td, hot):
    import trixilw_hip as tlw

    print(f"boundary split {kind} N={N} {td} {hot}", flush=True)
    semi, o, u0, mesh = case(oracle_mod, kind, N, td)
    lex = kind != "refined"
    E = len(u0)
    # an element with a boundary face, or one with none in the middle of the mesh
    nbr = mesh.neighbors[mesh.lexicographic_permutation()] if lex else mesh.neighbors
    at_bnd = (nbr == -1).any(axis=1)
    e = int(np.nonzero(at_bnd)[0][0]) if hot == "corner" else E // 2 + int(np.nonzero(~at_bnd[E // 2:])[0][0])
    u0 = with_hot_element(u0, e)
    K, cfl = 3, 0.2
    u_ref, t_ref, _ = o.solve(u0, 0.0, 1e9, cfl, max_steps=K, mdrk=td == "mdrk")
    u_dev = to_dev(mesh, u0) if lex else torch_mod().from_numpy(np.ascontiguousarray(u0)).cuda()
    # the workgroups with a boundary face, and not all of them
    assert 0 < launch_info(semi)[0] < E // (5 if N == 4 else 8)
    sol = run(semi, u_dev, K, tlw.CFLBased(cfl))
    assert sol.stats.naccept == K and abs(sol.t - t_ref) <= 1e-13 * t_ref
    assert_close(to_lex(mesh, sol.u) if lex else sol.u.cpu().numpy(), u_ref, what=f"{kind} N={N} {td} {hot}")
    semi.close()


# one workgroup below the line and on it
@pytest.mark.parametrize("N,nx,ny,split", [(3, 255, 128, False), (3, 256, 128, True), (4, 25, 819, False),
                                           (4, 160, 128, True)])
def test_split_line(oracle_mod, N, nx, ny, split):
    import trixilw_hip as tlw

    print(f"split line N={N} {nx}x{ny}", flush=True)
    semi, o, u0, mesh = setup_curved(oracle_mod, N, nx, ny, A=0.02, periodic=False)
    u_ref, t_ref, _ = o.solve(u0, 0.0, 1e9, 0.2, max_steps=1)
    assert (launch_info(semi)[0] > 0) == split
    sol = run(semi, to_dev(mesh, u0), 1, tlw.CFLBased(0.2))
    assert abs(sol.t - t_ref) <= 1e-13 * t_ref
    assert_close(to_lex(mesh, sol.u), u_ref, what=f"split line N={N} {nx}x{ny}")
    semi.close()


def test_split_adaptive_steps(oracle_mod):
    """The admissibility test of an adaptive step over both launches: from a dt that is far too
    large (rejected attempts) and from a small one."""
    import trixilw_hip as tlw

    torch_mod()
    print("split adaptive", flush=True)
    N, level, tol = 4, 8, {"abstol": 1e-6, "reltol": 1e-6}
    eq = tlw.CompressibleEulerEquations2D(1.4)
    ic = tlw.IsentropicVortex(center=(0.7, -0.4), period=(1e9, 1e9))
    mesh = tlw.TreeMesh((-10.0, -10.0), (10.0, 10.0), level, periodicity=False)
    solver = tlw.DGSEM(N)
    semi = tlw.SemidiscretizationHyperbolic(mesh, tlw.LW(), eq, ic, solver, boundary_conditions=ic)
    nx = mesh.nx
    o = oracle_mod.Oracle(N, nx, nx, -10.0, -10.0, 20.0 / nx, periodic=(False, False), bc_kind=ic.kind,
                          bc_par=ic.params, tolerances=(tol["abstol"], tol["reltol"]))
    x, y = o.node_coords()
    u0 = ic(x, y, 0.0) * (1.0 + 1e-4 * np.random.default_rng(2).standard_normal(x.shape + (4,)))
    tf = 0.05
    assert launch_info(semi)[0] > 0
    for dt0 in (1e-3, 1.0):
        u_ref, t_ref, dts, nrej = o.solve_adaptive(u0, 0.0, tf, dt0, max_attempts=500)
        sol = run(semi, to_dev(mesh, u0), None, tlw.Adaptive(), tf=tf, dt0=dt0, tol=tol)
        assert (sol.stats.naccept, sol.stats.nreject) == (len(dts), nrej)
        assert dt0 < tf or nrej > 0
        assert abs(sol.t - t_ref) <= 1e-13 * t_ref
        assert_close(to_lex(mesh, sol.u), u_ref, what=f"split adaptive dt0={dt0}")
    semi.close()
