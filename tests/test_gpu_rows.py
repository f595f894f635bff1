"""The x sweep along rows (k_rows_x: unequal widths, FP64, WENO5, one to three
fluids) against the FP64 oracle: rows of planes set end to end that fill the 58
columns of a wave exactly, one less and one more (52, 51 and 53 cells with six
ghost cells and these planes), rows that end inside a wave's columns, every
boundary code in x, 2D and 3D, RK2 and RK3.  Bars: the plain form bitwise,
right-hand side and step; the contracted form's step within 1e-12
(helpers.state_linf)."""
import numpy as np
import pytest

from microfc_amd import PREC_FP64, PREC_FP64_FAST, RhsModule, ic
from oracle import oracle as O

from helpers import (field_3d_case, multi_fluid_2d, one_fluid_3d_case, perturbed, say, state_linf, stretched_grids,
                     to_oracle)

pytestmark = pytest.mark.gpu


def _bubble(m, n, bc):
    prm, _, q = ic.shock_bubble_2d(N=620)
    prm.bc_beg, prm.bc_end = (bc[0], -3, -3), (bc[1], -4, -3)
    return prm, stretched_grids(prm), perturbed(prm, q)


def _fluids3():
    prm, _, q = multi_fluid_2d(3, N=601)
    prm.time_stepper = 2
    prm.bc_beg, prm.bc_end = (-4, -2, -3), (-2, -4, -3)
    return prm, stretched_grids(prm), q


def _one_fluid():
    prm, _, q = one_fluid_3d_case(69, 66, 62, (-1, -1, -1), (-1, -1, -1))
    return prm, stretched_grids(prm), q


CASES = {
    "2d_walls": lambda: _bubble(619, 619, (-2, -4)),
    "2d_three_fluids": _fluids3,
    "3d_52": lambda: field_3d_case(51, 89, 79, (-2, -4, -1), (-4, -2, -1), grid="stretched"),
    "3d_51": lambda: field_3d_case(50, 92, 77, (-3, -2, -4), (-2, -3, -4), grid="stretched", time_stepper=2),
    "3d_53": lambda: field_3d_case(52, 88, 78, (-1, -1, -2), (-1, -1, -2), grid="stretched"),
    "3d_one_fluid": _one_fluid,
}


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_FP64_FAST])
@pytest.mark.parametrize("name", list(CASES))
def test_rows_against_the_oracle(gpu, name, precision):
    torch = gpu
    prm, grids, q = CASES[name]()
    oc = to_oracle(prm)
    prm.precision = precision
    mod = RhsModule(prm, grids)
    try:
        qd = torch.from_numpy(q.copy()).cuda()
        q2, rd = mod.new_field(), mod.new_field(ghosted=False)
        mod.s_compute_rhs(qd, None, rd, 0)
        mod.sync()
        if precision == PREC_FP64:
            assert np.array_equal(rd.cpu().numpy(), O.compute_rhs(oc, grids, q))
        dt = mod.cfl_dt(qd, 0.3)
        mod.s_tvd_rk(0, (qd, q2), None, rd, dt)
        mod.sync()
        qo = q.copy()
        O.tvd_rk_step(oc, grids, dt, qo)
        got, want = prm.interior(qd.cpu().numpy()), prm.interior(qo)
        err = state_linf(prm, got, want, q)
        say(f"[rows] {name} precision {precision} {err.max():.2e}")
        if precision == PREC_FP64:
            assert np.array_equal(got, want)
        assert err.max() <= 1e-12
    finally:
        mod.finalize()
