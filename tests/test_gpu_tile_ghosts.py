"""Ghost cells that the sweeps fill while they write an RK stage, in the cases
that the RK stage in one kernel leaves to them: the fused x and y tile on 2D
grids too large for it (plain and contracted, every pair of boundary codes, one
and two fluids, RK2 and RK3), the x sweep on 1D grids too large for it, 1D and 2D runs of the FP32-bulk and learned forms
with one to four fluids.

A step against the FP64 oracle (the plain form bitwise, a contracted step within
1e-12, the others within 1e-3 of each variable's scale, as on other grids), and
the ghost cells of the last stage's input, which the step leaves in q_cons_ts(2),
bit for bit the oracle's boundary fill of its interior."""
import numpy as np
import pytest

from microfc_amd import PREC_FP32_BULK, PREC_FP32_LEARNED, PREC_FP64, PREC_FP64_FAST, RhsModule, ic, learned
from microfc_amd.rhs import Params
from oracle import oracle as O

from helpers import perturbed, say, state_linf, to_oracle
from test_gpu_stage_ghosts import BCS

pytestmark = pytest.mark.gpu


def _case(m, n, fluids, stepper, bx, by):
    gam = [4.4, 1.4, 1.667, 2.1][:fluids]
    pinf = [6e8, 0.0, 0.0, 1e5][:fluids] if fluids > 1 else [0.0]
    prm = Params(m=m, n=n, num_fluids=fluids, weno_order=5, time_stepper=stepper, gammas=[1 / (g - 1) for g in gam],
                 pi_infs=[g * p / (g - 1) for g, p in zip(gam, pinf)], bc_beg=(bx[0], by[0], -3), bc_end=(bx[1], by[1], -3))
    g = ic.uniform_grids(prm)
    X, Y, _ = ic.mesh(prm, g)
    Y = Y if n else 0.3 + 0 * X
    w = [1.0 + 0.5 * np.sin((7 + 2 * i) * X + 4 * Y + i) for i in range(fluids)]
    al = [x / sum(w) for x in w]
    vel = [30 + 40 * np.sin(7 * Y + X), 25 * np.cos(5 * X) + 20 * Y][:2 if n else 1]
    prim = np.stack([a * r for a, r in zip(al, (1000.0, 1.2, 0.2, 50.0))] + vel +
                    [1e6 * (1 + 0.3 * np.cos(11 * X - 3 * Y))] + al)
    return prm, g, perturbed(prm, ic.ghosted(prm, ic.prim_to_cons(prm, prim)), amp=1e-2)


def _step(torch, prm, grids, q, precision, variants, bc_fills):
    oc = to_oracle(prm)
    prm.precision = precision
    mod = RhsModule(prm, grids)
    try:
        qd = torch.from_numpy(q.copy()).cuda()
        q2, rd = mod.new_field(), mod.new_field(ghosted=False)
        dt = mod.cfl_dt(qd, 0.3)
        mod.timing(enable=True, reset=True)
        mod.s_tvd_rk(0, (qd, q2), None, rd, dt)
        mod.sync()
        assert mod.timing(enable=False)["bc_fill"][1] == bc_fills
        assert mod.timing_variants() == variants
        last = q2.cpu().numpy()
        assert np.array_equal(last, O.bc_fill(oc, last.copy()))
        qo = q.copy()
        O.tvd_rk_step(oc, grids, dt, qo)
        got, want = prm.interior(qd.cpu().numpy()), prm.interior(qo)
        err = state_linf(prm, got, want, q).max()
        say(f"[tile ghosts] {prm.m + 1}x{prm.n + 1} fluids {prm.num_fluids} bc {prm.bc_beg} {prm.bc_end} "
            f"precision {precision} {err:.2e}")
        if precision == PREC_FP64:
            assert np.array_equal(got, want)
        assert np.all(np.isfinite(got)) and err <= (1e-12 if precision in (PREC_FP64, PREC_FP64_FAST) else 1e-3)
    finally:
        mod.finalize()


@pytest.mark.parametrize("m,n,fluids,stepper,precision", [
    (255, 255, 2, 3, PREC_FP64), (511, 127, 1, 2, PREC_FP64), (255, 255, 2, 2, PREC_FP64_FAST),
    (299, 210, 2, 3, PREC_FP64_FAST), (211, 300, 1, 3, PREC_FP64_FAST)])
def test_fused_tile(gpu, m, n, fluids, stepper, precision):
    for bx, by in BCS:
        _step(gpu, *_case(m, n, fluids, stepper, bx, by), precision, {"tile_xy": stepper}, 1)


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_FP64_FAST])
@pytest.mark.parametrize("fluids", [1, 2])
def test_long_1d(gpu, fluids, precision):
    # more than 1600 tiles of 62 cells
    for bx, _ in BCS[2:]:
        _step(gpu, *_case(99999, 0, fluids, 3, bx, (-3, -3)), precision, {}, 1)


@pytest.mark.parametrize("precision", [PREC_FP32_BULK, PREC_FP32_LEARNED])
@pytest.mark.parametrize("fluids", [1, 2, 3, 4])
@pytest.mark.parametrize("m,n", [(130, 0), (62, 40)])
def test_single_precision_forms(gpu, m, n, fluids, precision):
    if precision == PREC_FP32_LEARNED:
        learned.Mlp()
    elif n:
        pytest.skip("FP32 bulk leaves the ghost cells of 2D stages to the boundary fill")
    for bx, by in BCS if n else sorted({(b[0], (-3, -3)) for b in BCS}):
        _step(gpu, *_case(m, n, fluids, 3, bx, by), precision, {}, 1)
