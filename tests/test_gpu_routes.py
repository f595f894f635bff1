"""Which kernel a sweep is (mfc_timing_read, ids 9 to 14) on the grids whose
results the other tests hold to the oracle: the marches, the x sweep along rows,
the fused tile and the RK stage in one kernel report under the direction's id
like the sweeps they stand in for, so a moved line could leave them untested.

The contracted right-hand side of the marches and of the rows against the oracle
too.  Bar: 16 roundings of the largest flux on both faces of the narrowest cell,
16 eps (|u| + c) Q / min(ds) summed over the directions, Q the variable's scale
(helpers.state_linf); 16 is twice the square root of the about 60 roundings
between the state and a face's flux."""
import numpy as np
import pytest

from microfc_amd import PREC_FP32_BULK, PREC_FP64, PREC_FP64_FAST, RhsModule, ic
from oracle import oracle as O

from helpers import multi_fluid_3d, perturbed, say, stretched_grids, to_oracle
from test_gpu_march import CASES as MARCH
from test_gpu_march import RUNS as MARCH_RUNS
from test_gpu_march_chunks import CASES as CHUNKS
from test_gpu_rows import CASES as ROWS
from test_gpu_stage_ghosts import _case

pytestmark = pytest.mark.gpu


def _three(n, stretched, bcb, bce):
    prm, grids, q = multi_fluid_3d(3, N=n)
    prm.bc_beg, prm.bc_end = bcb, bce
    return prm, stretched_grids(prm) if stretched else grids, perturbed(prm, q)


def _flat(nx, ny):
    return lambda: _case(nx - 1, ny - 1, 5, 3, (-2, -4), (-4, -2))


def _runs():
    out = []
    for name, p in MARCH_RUNS:
        out.append((f"march-{name}", MARCH[name], p, {"march_xy": 1, "march_z": 1} if "3d" in name else {"march_xy": 1}))
    for name, make in CHUNKS.items():
        for p in (PREC_FP64, PREC_FP64_FAST, PREC_FP32_BULK):
            out.append((f"chunks-{name}", make, p, {"march_xy": 1, "march_z": 1} if name == "3d" else {"march_xy": 1}))
    for p in (PREC_FP64, PREC_FP64_FAST):
        for name, make in ROWS.items():
            out.append((f"rows-{name}", make, p, {"rows_x": 1}))
        out.append(("fluids3-117", lambda: _three(117, True, (-2, -4, -3), (-4, -2, -2)), p,
                    {"rows_x": 1, "march_y": 1, "march_z": 1}))
        out.append(("fluids3-146", lambda: _three(146, False, (-3, -2, -1), (-2, -3, -1)), p,
                    {"rows_x": 1, "march_y": 1, "march_z": 1}))
        out.append(("tile-256", _flat(256, 256), p, {"tile_xy": 1}))
    return out


RUNS = _runs()


def _bar(prm, grids, q):
    nf, D, b = prm.num_fluids, prm.num_dims, prm.buff_size
    qi = np.asarray(prm.interior(q), dtype=np.float64)
    rho = sum(qi[i] for i in range(nf))
    gam = sum(qi[nf + D + 1 + i] * prm.gammas[i] for i in range(nf))
    pinf = sum(qi[nf + D + 1 + i] * prm.pi_infs[i] for i in range(nf))
    dyn = sum(0.5 * qi[nf + d] ** 2 for d in range(D)) / rho
    c = np.sqrt(((gam + 1.0) * (qi[nf + D] - dyn - pinf) / gam + pinf) / (gam * rho))
    Q = [np.max(np.abs(qi[i])) for i in range(nf)] + [np.max(rho) * np.max(c)] * D + [np.max(np.abs(qi[nf + D]))] + [1.0] * nf
    s = sum((np.max(np.abs(qi[nf + d] / rho)) + np.max(c)) / np.min(grids[d][1][b:-b]) for d in range(D))
    return 16 * np.finfo(np.float64).eps * s * np.array(Q)


@pytest.mark.parametrize("name,make,precision,kernels", RUNS, ids=[f"{r[0]}-{r[2]}" for r in RUNS])
def test_kernels_of_a_right_hand_side(gpu, name, make, precision, kernels):
    torch = gpu
    prm, grids, q = make()
    oc = to_oracle(prm)
    prm.precision = precision
    mod = RhsModule(prm, grids)
    try:
        qd = torch.from_numpy(q.copy()).cuda()
        rd = mod.new_field(ghosted=False)
        mod.timing(enable=True, reset=True)
        mod.s_compute_rhs(qd, None, rd, 0)
        mod.sync()
        mod.timing(enable=False)
        got = mod.timing_variants()
        say(f"[routes] {name} precision {precision} {got}")
        assert got == kernels
        if precision == PREC_FP64_FAST and not name.startswith("tile"):
            ref = O.compute_rhs(oc, grids, q)
            err = np.max(np.abs(rd.cpu().numpy() - ref).reshape(prm.sys_size, -1), axis=1) / _bar(prm, grids, q)
            say(f"[routes] {name} contracted right-hand side, parts of the bar {np.array2string(err, precision=3)}")
            assert err.max() <= 1.0
    finally:
        prm.precision = 0
        mod.finalize()


@pytest.mark.parametrize("nx,ny,precision,kernels", [(61, 1, PREC_FP64, {"stage": 3}), (63, 1, PREC_FP64_FAST, {"stage": 3}),
                                                     (256, 160, PREC_FP64, {"stage": 3}), (256, 161, PREC_FP64, {"tile_xy": 3}),
                                                     (256, 256, PREC_FP64_FAST, {"tile_xy": 3})])
def test_kernels_of_a_small_step(gpu, nx, ny, precision, kernels):
    torch = gpu
    prm, grids, q = _case(nx - 1, ny - 1, 5, 3, (-2, -4), (-1, -1))
    if ny == 160 or ny == 161:  # equal widths bit for bit
        b = prm.buff_size
        grids = [(np.arange(-b, n + b + 1) / 256.0, np.full(n + 2 * b, 1 / 256.0)) for n in (nx, ny)]
    prm.precision = precision
    mod = RhsModule(prm, grids)
    try:
        qd = torch.from_numpy(q.copy()).cuda()
        q2, rd = mod.new_field(), mod.new_field(ghosted=False)
        dt = mod.cfl_dt(qd, 0.3)
        mod.timing(enable=True, reset=True)
        mod.s_tvd_rk(0, (qd, q2), None, rd, dt)
        mod.sync()
        mod.timing(enable=False)
        assert mod.timing_variants() == kernels
    finally:
        mod.finalize()
