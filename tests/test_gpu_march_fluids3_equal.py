"""The z march with three fluids on equal widths (the y direction keeps its
tiles there): 128 x 96 x 256 cells, equal bit for bit, so the plain form takes it
too; walls, RK2 and RK3, against the FP64 oracle.  Bars: the plain form bitwise,
right-hand side and step; a contracted step within 1e-12 (helpers.state_linf)."""
import numpy as np
import pytest

from microfc_amd import PREC_FP64, PREC_FP64_FAST, RhsModule, ic
from microfc_amd.rhs import Params
from oracle import oracle as O

from helpers import perturbed, say, state_linf, to_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stepper,bcb,bce", [(3, (-2, -4, -3), (-4, -2, -2)), (2, (-1, -1, -4), (-1, -1, -2))])
def test_three_fluids_on_equal_widths(gpu, stepper, bcb, bce):
    torch = gpu
    gam, pinf = (4.4, 1.4, 1.667), (6e8, 0.0, 0.0)
    prm = Params(m=127, n=95, p=255, num_fluids=3, weno_order=5, time_stepper=stepper, gammas=[1 / (g - 1) for g in gam],
                 pi_infs=[g * p / (g - 1) for g, p in zip(gam, pinf)], bc_beg=bcb, bc_end=bce)
    grids = ic.uniform_grids(prm, hi=(1.0, 0.75, 2.0))
    X, Y, Z = ic.mesh(prm, grids)
    w = [1.0 + 0.5 * np.sin((5 + 2 * i) * X + i) * np.cos(3 * Y - 2 * Z + i) for i in range(3)]
    al = [x / sum(w) for x in w]
    prim = np.stack([a * r for a, r in zip(al, (1000.0, 1.2, 0.2))] +
                    [10 * np.sin(6 * Y) + 0 * X, 5 * np.cos(6 * X) * np.sin(3 * Y), 3 * np.sin(6 * (X + Z)),
                     1e5 * (1 + 0.5 * np.exp(-((X - 0.4) ** 2 + (Y - 0.4) ** 2 + (Z - 1) ** 2) / 0.02))] + al)
    q = perturbed(prm, ic.ghosted(prm, ic.prim_to_cons(prm, prim)))
    oc = to_oracle(prm)
    ref, step = O.compute_rhs(oc, grids, q), None
    for precision in (PREC_FP64, PREC_FP64_FAST):
        prm.precision = precision
        mod = RhsModule(prm, grids)
        try:
            qd = torch.from_numpy(q.copy()).cuda()
            q2, rd = mod.new_field(), mod.new_field(ghosted=False)
            mod.timing(enable=True, reset=True)
            mod.s_compute_rhs(qd, None, rd, 0)
            mod.sync()
            mod.timing(enable=False)
            assert mod.timing_variants() == {"march_z": 1}
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
            say(f"[march 3 fluids, equal widths] precision {precision} {err.max():.2e}")
            if precision == PREC_FP64:
                assert np.array_equal(got, want)
            assert err.max() <= 1e-12
        finally:
            prm.precision = 0
            mod.finalize()
