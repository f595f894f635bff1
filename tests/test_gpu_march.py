"""The marching sweeps (k_march), which take over from the tile kernels and
the separate sweeps on large grids, against the FP64 oracle: cell counts that
leave partial column sets and chunks, every boundary code in every direction,
equal and unequal cell widths, one and two fluids, RK2 and RK3.

Bars: the plain form is bitwise the oracle, right-hand side and step; the
contracted form's state one RK step from the oracle's own is within 1e-12
(helpers.state_linf; its right-hand side, a difference of fluxes over cell
widths of 1/100 and less, is 1.5e-12 off here, and 1.7e-12 in the kernels
these replace, so it carries no bar); the FP32-bulk form is within 1e-3 of each
variable's scale, as on small grids."""
import numpy as np
import pytest

from microfc_amd import PREC_FP32_BULK, PREC_FP64, PREC_FP64_FAST, RhsModule, ic
from oracle import oracle as O

from helpers import field_3d_case, one_fluid_3d_case, perturbed, say, scaled_linf, state_linf, stretched_grids, to_oracle

pytestmark = pytest.mark.gpu


def _stretched_2d():
    prm, _, q = ic.shock_bubble_2d(N=1237)
    prm.bc_beg, prm.bc_end = (-2, -4, -3), (-4, -2, -3)
    return prm, stretched_grids(prm), perturbed(prm, q)


def _uniform_2d():
    # 2048 x 4104 cells: a wave's entries span the ends of row chunks
    prm = ic.shock_bubble_2d(N=64)[0]
    prm.m, prm.n, prm.time_stepper = 2047, 4103, 2
    prm.bc_beg, prm.bc_end = (-1, -4, -3), (-1, -2, -3)
    g = ic.uniform_grids(prm)
    X, Y, _ = ic.mesh(prm, g)
    a = 0.5 + 0.4 * np.sin(9 * X + 4 * Y)
    prim = np.stack([1000 * a, 1.2 * (1 - a), 30 * np.sin(7 * Y), 20 * np.cos(5 * X) * Y,
                     1e6 * (1 + 0.3 * np.cos(11 * X - 3 * Y)), a, 1 - a])
    return prm, g, perturbed(prm, ic.ghosted(prm, ic.prim_to_cons(prm, prim)))


CASES = {
    "stretched_2d_walls": _stretched_2d,
    "uniform_2d_rk2": _uniform_2d,
    "stretched_3d_walls": lambda: field_3d_case(126, 98, 121, (-2, -4, -1), (-4, -2, -1), grid="stretched"),
    "stretched_3d_riemann_z": lambda: field_3d_case(140, 70, 155, (-1, -3, -4), (-1, -2, -2), grid="stretched",
                                                    time_stepper=2),
    "uniform_3d_walls": lambda: field_3d_case(127, 127, 191, (-4, -2, -2), (-2, -4, -4)),
    "uniform_3d_one_fluid": lambda: one_fluid_3d_case(127, 127, 191, (-1, -1, -1), (-1, -1, -1)),
}
RUNS = [(c, p) for c in CASES for p in (PREC_FP64, PREC_FP64_FAST)] + [
    (c, PREC_FP32_BULK) for c in ("stretched_2d_walls", "stretched_3d_walls")]


def _kernels(mod):
    return {k: v[1] for k, v in mod.timing(enable=False).items() if v[1]}


@pytest.mark.parametrize("name,precision", RUNS, ids=[f"{c}-{p}" for c, p in RUNS])
def test_march_against_the_oracle(gpu, name, precision):
    torch = gpu
    prm, grids, q = CASES[name]()
    oc = to_oracle(prm)
    ref = O.compute_rhs(oc, grids, q)
    prm.precision = precision
    mod = RhsModule(prm, grids)
    try:
        qd = torch.from_numpy(q.copy()).cuda()
        rd = mod.new_field(ghosted=False)
        mod.timing(enable=True, reset=True)
        mod.s_compute_rhs(qd, None, rd, 0)
        mod.sync()
        # the x and y directions in one launch: on unequal widths only the
        # march does that
        assert _kernels(mod).get("sweep_xy") == 1
        got = rd.cpu().numpy()
        err = scaled_linf(prm, got, ref)
        say(f"[march] {name} precision {precision} rhs {np.array2string(err, precision=2)}")
        assert np.all(np.isfinite(got))
        if precision == PREC_FP64:
            assert np.array_equal(got, ref)
        if precision == PREC_FP32_BULK:
            assert err.max() <= 1e-3
        dt = mod.cfl_dt(qd, 0.3)
        q2 = mod.new_field()
        mod.s_tvd_rk(0, (qd, q2), None, rd, dt)
        mod.sync()
        got = prm.interior(qd.cpu().numpy())
        qo = q.copy()
        O.tvd_rk_step(oc, grids, dt, qo)
        want = prm.interior(qo)
        err = state_linf(prm, got, want, q)
        say(f"[march] {name} precision {precision} step {np.array2string(err, precision=2)}")
        if precision == PREC_FP64:
            assert np.array_equal(got, want)
        # FP32: three stages, each adding at most dt times its right-hand
        # side's error of 1e-3 of a scale that changes by less than itself
        assert err.max() <= (1e-3 if precision == PREC_FP32_BULK else 1e-12)
    finally:
        prm.precision = 0
        mod.finalize()
