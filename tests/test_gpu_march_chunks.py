"""Marches in chunks of few rows (8 to 15, which grids just above the marches'
sizes take so that every wave has a place at once), the last chunk one row,
against the FP64 oracle: 1281 x 1171 cells (13 rows a chunk in FP64, 9 in FP32)
and 129 x 118 x 100 (9 rows along y and z in FP32), unequal widths.  Bars as for
the marches in larger chunks: the plain form bitwise, right-hand side and step;
a contracted step within 1e-12, FP32 bulk within 1e-3 (helpers.state_linf)."""
import numpy as np
import pytest

from microfc_amd import PREC_FP32_BULK, PREC_FP64, PREC_FP64_FAST, RhsModule, ic
from oracle import oracle as O

from helpers import field_3d_case, perturbed, say, scaled_linf, state_linf, stretched_grids, to_oracle

pytestmark = pytest.mark.gpu


def _flat():
    prm = ic.shock_bubble_2d(N=64)[0]
    prm.m, prm.n = 1280, 1170
    prm.bc_beg, prm.bc_end = (-2, -4, -3), (-4, -2, -3)
    X, Y, _ = ic.mesh(prm, ic.uniform_grids(prm))
    a = 0.5 + 0.4 * np.sin(9 * X + 4 * Y)
    prim = np.stack([1000 * a, 1.2 * (1 - a), 30 * np.sin(7 * Y + X), 20 * np.cos(5 * X) * Y,
                     1e6 * (1 + 0.3 * np.cos(11 * X - 3 * Y)), a, 1 - a])
    return prm, stretched_grids(prm), perturbed(prm, ic.ghosted(prm, ic.prim_to_cons(prm, prim)))


CASES = {"2d": _flat, "3d": lambda: field_3d_case(128, 117, 99, (-2, -4, -1), (-4, -2, -1), grid="stretched")}


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_FP64_FAST, PREC_FP32_BULK])
@pytest.mark.parametrize("name", list(CASES))
def test_short_chunks(gpu, name, precision):
    torch = gpu
    prm, grids, q = CASES[name]()
    oc = to_oracle(prm)
    ref = O.compute_rhs(oc, grids, q)
    prm.precision = precision
    mod = RhsModule(prm, grids)
    try:
        qd = torch.from_numpy(q.copy()).cuda()
        q2, rd = mod.new_field(), mod.new_field(ghosted=False)
        mod.timing(enable=True, reset=True)
        mod.s_compute_rhs(qd, None, rd, 0)
        mod.sync()
        # x and y in one launch on unequal widths: the march
        assert mod.timing(enable=False)["sweep_xy"][1] == 1
        got = rd.cpu().numpy()
        if precision == PREC_FP64:
            assert np.array_equal(got, ref)
        elif precision == PREC_FP32_BULK:
            assert scaled_linf(prm, got, ref).max() <= 1e-3
        dt = mod.cfl_dt(qd, 0.3)
        mod.s_tvd_rk(0, (qd, q2), None, rd, dt)
        mod.sync()
        qo = q.copy()
        O.tvd_rk_step(oc, grids, dt, qo)
        got, want = prm.interior(qd.cpu().numpy()), prm.interior(qo)
        err = state_linf(prm, got, want, q)
        say(f"[march chunks] {name} precision {precision} {err.max():.2e}")
        if precision == PREC_FP64:
            assert np.array_equal(got, want)
        assert err.max() <= (1e-3 if precision == PREC_FP32_BULK else 1e-12)
    finally:
        mod.finalize()
