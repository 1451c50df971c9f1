"""solve_lwfr's device loop from any form of the initial state it accepts: a contiguous
device tensor, a view with other strides and a host tensor give the same bits."""
import numpy as np
import pytest

from gpu_helpers import setup, torch_mod

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
