"""Viscous runs at the edges of the kernels' tiles (62 cells of a row in x,
16 x 14 cells in y, 32 x 8 ghosted cells of the gradient pass, 256 in 1D):
whole tiles, one cell less and one more, every boundary code, equal and unequal
widths, finite-difference and reconstructed gradients, one to four fluids.
Bar: relative L-infinity 1e-12 per step against the FP64 oracle, as for the
other viscous cases."""
import numpy as np
import pytest

from microfc_amd import RhsModule, ic
from oracle import oracle as O

from helpers import assert_parity, multi_fluid_2d, perturbed, relayout, say, stretched_grids, to_oracle

pytestmark = pytest.mark.gpu

SIZES = [(61, 27, (-3, -4), (-2, -3), False), (62, 28, (-4, -4), (-4, -4), True), (124, 26, (-2, -4), (-2, -2), False),
         (249, 0, (-4, -3), (-3, -3), False), (123, 69, (-1, -1), (-1, -1), True)]


@pytest.mark.parametrize("wrf", [False, True])
@pytest.mark.parametrize("fluids", [1, 2, 4])
@pytest.mark.parametrize("m,n,bcx,bcy,stretch", SIZES)
def test_viscous_tile_edges(gpu, m, n, bcx, bcy, stretch, fluids, wrf):
    torch = gpu
    prm = multi_fluid_2d(fluids, N=32)[0]
    prm.m, prm.n = m, n
    prm.bc_beg, prm.bc_end = (bcx[0], bcy[0], -3), (bcx[1], bcy[1], -3)
    g = stretched_grids(prm) if stretch else ic.uniform_grids(prm)
    X = ic.mesh(prm, g)[0]
    Y = ic.mesh(prm, g)[1] if n else 0.3 + 0 * X
    al = [np.full_like(X, 1.0)] if fluids == 1 else [
        (1.0 + 0.5 * np.sin((3 + 2 * i) * X + (1 + i) * Y)) for i in range(fluids)]
    tot = sum(al)
    al = [x / tot for x in al]
    prim = np.stack([(1.0 + 0.4 * i) * al[i] for i in range(fluids)] +
                    [0.3 * np.sin(5 * X + Y), 0.2 * np.cos(4 * Y - X)][:2 if n else 1] +
                    [1.0 + 0.2 * np.cos(6 * X + 2 * Y)] + al)
    q = perturbed(prm, ic.ghosted(prm, ic.prim_to_cons(prm, prim)))
    prm.Re = [(20.0 + 5 * i, 30.0 if i % 2 == 0 else -1.0) for i in range(fluids)]
    prm.weno_Re_flux = wrf
    g, q = relayout(prm, g, q)
    oc = to_oracle(prm)
    mod = RhsModule(prm, g)
    try:
        say(f"[viscous tiles] {m + 1}x{n + 1} bc {bcx} {bcy} fluids {fluids} weno_Re_flux {wrf}")
        qd = torch.from_numpy(q.copy()).cuda()
        q2, rd = mod.new_field(), mod.new_field(ghosted=False)
        dt = 0.2 * mod.cfl_dt(qd, 1.0)
        mod.s_tvd_rk(0, (qd, q2), None, rd, dt)
        mod.sync()
        qo = q.copy()
        O.tvd_rk_step(oc, g, dt, qo)
        assert_parity(prm.interior(qd.cpu().numpy()), prm.interior(qo), what="step")
    finally:
        mod.finalize()
