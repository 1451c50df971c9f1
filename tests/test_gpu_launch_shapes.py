"""The rules that choose a launch by the mesh: the default tile of the volume
kernel, the surface launch split at the domain boundary, and the shock-capturing
workgroups with and without a blended element, each at its edges and against the
CPU oracle (1e-12 relative, the bound of the other parity tests; another order
of the same sums).  Inputs are seeded."""
import numpy as np
import pytest

from gpu_helpers import assert_close, setup, setup_curved, to_dev, to_lex, torch_mod
from test_gpu_curved_sc_parity import with_jump

pytestmark = pytest.mark.gpu


def rhs_pair(semi, o, mesh, u_lex, cfl):
    import trixilw_hip as tlw

    torch = torch_mod()
    dt = cfl * o.max_dt(u_lex)
    ref = o.rhs(u_lex, 0.0, dt)
    u = to_dev(mesh, u_lex)
    du = torch.empty_like(u)
    semi.cache["dt"][0] = dt
    tlw.rhs(du, u, semi, 0.0)
    torch.cuda.synchronize()
    return to_lex(mesh, du), ref


# the sizes on both sides of each line of the rule, with ragged last workgroups
@pytest.mark.parametrize("N,nx,ny,tile", [(3, 64, 32, 4), (3, 683, 3, 8), (3, 256, 128, 8), (3, 331, 99, 16),
                                          (4, 128, 128, 5), (4, 145, 113, 10)])
def test_default_tile(oracle_mod, N, nx, ny, tile):
    print(f"default tile N={N} {nx}x{ny}", flush=True)
    semi, o, u_lex, mesh = setup_curved(oracle_mod, N, nx, ny, A=0.02)
    assert semi.elements_per_workgroup() == tile
    du, ref = rhs_pair(semi, o, mesh, u_lex, 0.4)
    assert_close(du, ref, what=f"N={N} {nx}x{ny}")
    semi.close()


# from 4096 workgroups on (5 elements each for N=4, 8 for N=3) the elements with a
# boundary face are launched apart: a level below that, and the first one above it
@pytest.mark.parametrize("N,level", [(3, 7), (3, 8), (4, 7), (4, 8)])
@pytest.mark.parametrize("ordering", ["strips", "morton"])
def test_boundary_surface_launch(oracle_mod, N, level, ordering):
    import trixilw_hip as tlw

    print(f"boundary launch N={N} level={level} {ordering}", flush=True)
    ic = tlw.FourQuadrantRiemann()
    semi, o, u_lex, mesh = setup(oracle_mod, N, level, periodic=False, domain=(0.0, 1.0), bc=ic, ic=ic, amp=1e-3,
                                 keep_aux=False, ordering=ordering)
    du, ref = rhs_pair(semi, o, mesh, u_lex, 0.05)
    assert_close(du, ref, what=f"N={N} level={level} {ordering}")
    semi.close()


# a few blended elements: at every tile some workgroups have one and some have none
@pytest.mark.parametrize("N,tile", [(3, 4), (3, 8), (3, 16), (4, 5), (4, 10), (4, 15)])
@pytest.mark.parametrize("mesh_kind", ["tree", "curved"])
def test_blended_and_pure_workgroups(oracle_mod, N, tile, mesh_kind):
    import trixilw_hip as tlw

    print(f"blended and pure workgroups {mesh_kind} N={N} tile={tile}", flush=True)
    if mesh_kind == "tree":
        ic = tlw.FourQuadrantRiemann()
        semi, o, u_lex, mesh = setup(oracle_mod, N, 6, periodic=False, domain=(0.0, 1.0), bc=ic, ic=ic, amp=0.0,
                                     sc=True, keep_aux=True)
    else:
        semi, o, u_lex, mesh = setup_curved(oracle_mod, N, 37, 29, A=0.05, sc=True, keep_aux=True)
        u_lex = with_jump(o, u_lex)
    semi.elements_per_workgroup(tile)
    du, ref = rhs_pair(semi, o, mesh, u_lex, 0.3)
    alpha = semi.get_aux("alpha")
    blended = [bool(np.any(alpha[k:k + tile] > 0.0)) for k in range(0, len(alpha), tile)]
    assert any(blended) and not all(blended)
    assert_close(du, ref, what=f"{mesh_kind} N={N} tile={tile}")
    semi.close()


# MDRK has its own line: one element below it and on it, both stages against the oracle
@pytest.mark.parametrize("N,nx,ny,tile", [(3, 16, 5, 8), (3, 127, 129, 8), (3, 128, 128, 16), (4, 128, 128, 5),
                                          (4, 145, 113, 10)])
def test_default_tile_mdrk(oracle_mod, N, nx, ny, tile):
    import trixilw_hip as tlw

    torch = torch_mod()
    print(f"default MDRK tile N={N} {nx}x{ny}", flush=True)
    semi, o, u_lex, mesh = setup_curved(oracle_mod, N, nx, ny, A=0.02, td="mdrk")
    assert semi.elements_per_workgroup() == tile
    dt = 0.2 * o.max_dt(u_lex)
    ref1 = o.rhs(u_lex, 0.0, dt, kind="mdrk1")
    us = u_lex + dt * ref1
    o.set_us(us)
    ref2 = o.rhs(u_lex, 0.0, dt, kind="mdrk2")
    u = to_dev(mesh, u_lex)
    du = torch.empty_like(u)
    semi.cache["dt"][0] = dt
    tlw.rhs_mdrk1(du, u, semi, 0.0)
    assert_close(to_lex(mesh, du), ref1, what=f"MDRK stage 1 N={N} {nx}x{ny}")
    semi.set_us(to_dev(mesh, us))
    tlw.rhs_mdrk2(du, u, semi, 0.0)
    assert_close(to_lex(mesh, du), ref2, what=f"MDRK stage 2 N={N} {nx}x{ny}")
    semi.close()
