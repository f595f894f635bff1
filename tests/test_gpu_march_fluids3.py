"""The y and z marches with three fluids, which take over from the separate
sweeps on large 3D grids (unequal widths; z also on equal widths): cell counts
that leave partial column sets and chunks, walls, RK2 and RK3, against the FP64
oracle.  Bars: the plain form bitwise, right-hand side and step; the contracted
form's step within 1e-12 and the FP32-bulk form's within 1e-3 (helpers.state_linf),
as for the marches with one and two fluids."""
import numpy as np
import pytest

from microfc_amd import PREC_FP32_BULK, PREC_FP64, PREC_FP64_FAST, RhsModule
from oracle import oracle as O

from helpers import multi_fluid_3d, perturbed, say, state_linf, stretched_grids, to_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,stretched,stepper,bcb,bce,precisions", [
    (117, True, 3, (-2, -4, -3), (-4, -2, -2), (PREC_FP64, PREC_FP64_FAST, PREC_FP32_BULK)),
    (131, True, 2, (-1, -1, -4), (-1, -1, -2), (PREC_FP64, PREC_FP64_FAST)),
    (146, False, 3, (-3, -2, -1), (-2, -3, -1), (PREC_FP64, PREC_FP64_FAST)),
])
def test_three_fluids_march(gpu, n, stretched, stepper, bcb, bce, precisions):
    torch = gpu
    prm, grids, q = multi_fluid_3d(3, N=n)
    prm.time_stepper, prm.bc_beg, prm.bc_end = stepper, bcb, bce
    if stretched:
        grids = stretched_grids(prm)
    q = perturbed(prm, q)
    oc = to_oracle(prm)
    ref = O.compute_rhs(oc, grids, q)
    step = None
    for precision in precisions:
        prm.precision = precision
        mod = RhsModule(prm, grids)
        try:
            qd = torch.from_numpy(q.copy()).cuda()
            q2, rd = mod.new_field(), mod.new_field(ghosted=False)
            mod.s_compute_rhs(qd, None, rd, 0)
            mod.sync()
            if precision == PREC_FP64:
                assert np.array_equal(rd.cpu().numpy(), ref)
            if step is None:
                dt = mod.cfl_dt(qd, 0.3)
                step = q.copy()
                O.tvd_rk_step(oc, grids, dt, step)
            mod.s_tvd_rk(0, (qd, q2), None, rd, dt)
            mod.sync()
            got, want = prm.interior(qd.cpu().numpy()), prm.interior(step)
            err = state_linf(prm, got, want, q)
            say(f"[march 3 fluids] {n}^3 stretched {stretched} precision {precision} {err.max():.2e}")
            if precision == PREC_FP64:
                assert np.array_equal(got, want)
            assert err.max() <= (1e-3 if precision == PREC_FP32_BULK else 1e-12)
        finally:
            prm.precision = 0
            mod.finalize()
