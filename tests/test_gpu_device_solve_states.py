"""solve_lwfr's device loop from any form of the initial state it accepts: a contiguous
device tensor, a view with other strides and a host tensor give the same bits."""
import numpy as np
import pytest

from gpu_helpers import launch_info, setup, torch_mod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,level", [(3, 2), (4, 2), (4, 3)])
@pytest.mark.parametrize("form", ["strided", "host"])
def test_solve_from_other_state_forms(oracle_mod, N, level, form):
    import trixilw_hip as tlw
    from trixilw_hip import _lib

    torch = torch_mod()
    semi, o, u_lex, mesh = setup(oracle_mod, N, level)
    lw_update = tlw.semidiscretize(semi, tlw.LW(), (0.0, 1e9))
    tsc = tlw.CFLBased(tlw.trixi2lw(0.9, semi.solver))
    ref = tlw.solve_lwfr(lw_update, (), 1e-6, None, time_step_computation=tsc, max_steps=3)
    u0 = lw_update.u0
    if form == "strided":
        wide = torch.empty((*u0.shape[:-1], 8), dtype=u0.dtype, device=u0.device)
        wide[..., ::2] = u0
        lw_update.u0 = wide[..., ::2]
    else:
        lw_update.u0 = u0.cpu()
    sol = tlw.solve_lwfr(lw_update, (), 1e-6, None, time_step_computation=tsc, max_steps=3)
    assert sol.u.is_cuda and sol.t == ref.t
    assert np.array_equal(sol.u.cpu().numpy(), ref.u.cpu().numpy())
    lw_update.u0 = u0[:-1]
    with pytest.raises(_lib.TLWError):
        tlw.solve_lwfr(lw_update, (), 1e-6, None, time_step_computation=tsc, max_steps=3)
    semi.close()


def test_solves_to_many_final_times_share_one_graph(oracle_mod):
    """With graph replay on, solves of different lengths capture the regular chunk alone (the step
    counts left at the end differ) and give the bits of launched steps; a count asked for again is
    captured too and replays to the same bits."""
    import trixilw_hip as tlw
    from trixilw_hip import _lib

    torch = torch_mod()
    semi, o, u_lex, mesh = setup(oracle_mod, 3, 3)
    tsc = tlw.CFLBased(tlw.trixi2lw(0.9, semi.solver))
    dt = tlw.trixi2lw(0.9, semi.solver) * o.max_dt(u_lex)
    stream = torch.cuda.Stream()
    times = [(8 + r) * dt for r in (1.5, 2.5, 3.5, 4.5, 5.5)]

    def solve(t_final):
        lw_update = tlw.semidiscretize(semi, tlw.LW(), (0.0, t_final))
        with torch.cuda.stream(stream):
            return tlw.solve_lwfr(lw_update, (), 1e-6, None, time_step_computation=tsc, chunk=8)

    ref = [solve(t) for t in times]
    _lib.check(_lib.lib().tlw_enable_graphs(semi.handle, 1), semi.handle)
    got = [solve(t) for t in times]
    assert launch_info(semi)[1] == 1
    assert len({s.stats.naccept for s in ref}) == len(times)
    again = [solve(times[0]) for _ in range(3)]
    assert launch_info(semi)[1] == 2
    for a, b in zip(got + again, ref + [ref[0]] * 3):
        assert a.t == b.t and a.stats.naccept == b.stats.naccept
        assert np.array_equal(a.u.cpu().numpy(), b.u.cpu().numpy())
    semi.close()
