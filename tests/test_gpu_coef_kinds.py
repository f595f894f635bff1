"""WENO5 coefficients in the contracted form: grids whose cells all have the
equal-width coefficients within 5e-13 run kernels with those constants built
in; grids whose cells have equal coefficients but others (geometric widths) run
the same kernels with the first cell's, not each cell's own.  Geometric grids
are compared with the FP64 oracle over every kernel that takes such a direction:
the RK stage in one kernel, the fused tile, the marches, the separate sweeps of
three fluids, 1D, and a grid geometric in one direction only.

Bar: a step within 1e-12 of the oracle (helpers.state_linf), the form's own."""
import numpy as np
import pytest

from microfc_amd import PREC_FP64_FAST, RhsModule, ic
from microfc_amd.rhs import uniform_cell_boundaries
from oracle import oracle as O

from helpers import field_3d_case, multi_fluid_3d, perturbed, say, state_linf, to_oracle

pytestmark = pytest.mark.gpu

CANON = np.array([1 / 3, -5 / 6, -1 / 6, -1 / 3, -2 / 3, 1 / 6, -1 / 6, 2 / 3, 1 / 3, 1 / 6, 5 / 6, -1 / 3, 0.1, 0.6, 0.3,
                  0.3, 0.6, 0.1, 4 / 3, -11 / 3, 10 / 3, 4 / 3, -5 / 3, 4 / 3, 10 / 3, -11 / 3, 4 / 3])[:, None]


def _geometric(s, b, ratio):
    """s_cb(-1-b..s+b) and ds(-b..s+b) of cells whose widths grow by one factor
    per cell, `ratio` over the whole direction, the ghost cells' too."""
    i = np.arange(-b, s + 2 + b).astype(np.longdouble)
    cb = (np.longdouble(ratio) ** (i / (s + 1)) - 1) / (np.longdouble(ratio) - 1)
    return cb.astype(np.float64), np.diff(cb.astype(np.float64))


def _kinds(cb, s, b):
    """Largest distance of a reconstructed cell's coefficients from the first's,
    and of the first's and of any cell's from the equal-width ones."""
    c = O.weno_coefficients(cb, s, b, 5)[:, b - 1:b + s + 2]
    return (np.max(np.abs(c / c[:, :1] - 1)), np.max(np.abs(c[:, :1] / CANON - 1)), np.max(np.abs(c / CANON - 1)))


def _bubble(m, n):
    prm = ic.shock_bubble_2d(N=64)[0]
    prm.m, prm.n = m, n
    prm.bc_beg, prm.bc_end = (-2, -4, -3) if n else (-2, -3, -3), (-4, -2, -3) if n else (-4, -3, -3)
    g = ic.uniform_grids(prm)
    X, Y = ic.mesh(prm, g)[0], ic.mesh(prm, g)[1] if n else 0.0
    a = 0.5 + 0.4 * np.sin(9 * X + 4 * Y)
    vel = [30 * np.sin(7 * Y + X), 20 * np.cos(5 * X) + 0 * Y][:2 if n else 1]
    prim = np.stack([1000 * a, 1.2 * (1 - a), *vel, 1e6 * (1 + 0.3 * np.cos(11 * X - 3 * Y)), a, 1 - a])
    return prm, perturbed(prm, ic.ghosted(prm, ic.prim_to_cons(prm, prim)))


def _field3d(m, n, p):
    prm, _, q = field_3d_case(m, n, p, (-2, -4, -1), (-4, -2, -1))
    return prm, q


def _three(N):
    prm, _, q = multi_fluid_3d(3, N=N)
    return prm, perturbed(prm, q)


CASES = {  # case, ratio of each direction, sweeps of one right-hand side
    "stage_1d": (lambda: _bubble(300, 0), (3.0,), {"sweep_x": 1}),
    "stage_2d": (lambda: _bubble(60, 47), (3.0, 0.5), {"sweep_xy": 1}),
    "tile_2d": (lambda: _bubble(299, 210), (2.0, 3.0), {"sweep_xy": 1}),
    "tile_2d_x_only": (lambda: _bubble(254, 255), (3.0, 1.0), {"sweep_xy": 1}),
    "march_2d": (lambda: _bubble(500, 16383), (2.0, 1.0), {"sweep_xy": 1}),
    "tile_3d": (lambda: _field3d(47, 39, 30), (2.0, 3.0, 0.5), {"sweep_xy": 1, "sweep_z": 1}),
    "march_3d": (lambda: _field3d(130, 150, 160), (2.0, 3.0, 0.5), {"sweep_xy": 1, "sweep_z": 1}),
    "three_fluids_3d": (lambda: _three(48), (2.0, 3.0, 0.5), {"sweep_x": 1, "sweep_y": 1, "sweep_z": 1}),
}


@pytest.mark.parametrize("name", list(CASES))
def test_geometric_grids(gpu, name):
    torch = gpu
    make, ratios, sweeps = CASES[name]
    prm, q = make()
    b = prm.buff_size
    grids = []
    for d, s in enumerate(prm.extents()):
        cb, ds = _geometric(s, b, ratios[d]) if ratios[d] != 1.0 else ic.uniform_grids(prm)[d]
        dev, _, far = _kinds(cb, s, b)
        assert dev <= 5e-13 and (far > 1e-4) == (ratios[d] != 1.0), (dev, far)
        grids.append((cb, ds))
    oc = to_oracle(prm)
    prm.precision = PREC_FP64_FAST
    mod = RhsModule(prm, grids)
    try:
        qd = torch.from_numpy(q.copy()).cuda()
        q2, rd = mod.new_field(), mod.new_field(ghosted=False)
        mod.timing(enable=True, reset=True)
        mod.s_compute_rhs(qd, None, rd, 0)
        mod.sync()
        n = {k: v[1] for k, v in mod.timing(enable=False).items() if v[1] and k.startswith("sweep")}
        assert n == sweeps
        dt = mod.cfl_dt(qd, 0.3)
        mod.s_tvd_rk(0, (qd, q2), None, rd, dt)
        mod.sync()
        qo = q.copy()
        O.tvd_rk_step(oc, grids, dt, qo)
        err = state_linf(prm, prm.interior(qd.cpu().numpy()), prm.interior(qo), q)
        say(f"[coef kinds] {name} {np.array2string(err, precision=2)}")
        assert err.max() <= 1e-12
    finally:
        mod.finalize()


def _drifting(s, b, a):
    """Boundaries whose widths grow by a factor 1 + a per cell at one end and 1
    + 2a at the other."""
    i = np.arange(-b, s + 2 + b).astype(np.longdouble)
    w = np.exp(np.longdouble(a) * (i + i * i / (2 * (s + 2 * b)))) / (s + 1)
    return np.concatenate([[-w[:b].sum()], -w[:b].sum() + np.cumsum(w[:-1])]).astype(np.float64)


@pytest.mark.parametrize("a,built_in", [(1e-14, True), (1e-13, False)])
def test_built_in_coefficients_are_within_the_tolerance(gpu, a, built_in):
    """x coefficients that drift from cell to cell: as long as every one is
    within 5e-13 of the equal-width ones the right-hand side is bitwise that of
    the equal-width grid (the widths passed are the same), and where one is
    farther, though the first is not and all are near the first, it is not."""
    torch = gpu
    prm, q = _bubble(63, 63)
    s, b = prm.m, prm.buff_size
    g = ic.uniform_grids(prm)
    cb = _drifting(s, b, a)
    near, first, far = _kinds(cb, s, b)
    say(f"[coef kinds] drift {a}: from the first {near:.1e}, the first {first:.1e} and the farthest {far:.1e} from equal widths")
    assert near <= 5e-13 and first <= 5e-13 and (far <= 5e-13) == built_in
    out = []
    prm.precision = PREC_FP64_FAST
    for grids in (g, [(cb, g[0][1]), g[1]]):
        mod = RhsModule(prm, grids)
        try:
            rd = mod.new_field(ghosted=False)
            mod.s_compute_rhs(torch.from_numpy(q.copy()).cuda(), None, rd, 0)
            mod.sync()
            out.append(rd.cpu().numpy())
        finally:
            mod.finalize()
    assert np.array_equal(*out) == built_in
