"""A right-hand side of the plain form whose primitive field comes from the x
and y march (interior) and the ghost fill (ghost cells) against the FP64
oracle, bitwise: right-hand side, the whole primitive field with edges and
corners, and the filled ghost cells of the input; every boundary code, equal
and unequal widths, one and two fluids, 2D and 3D, cell counts that leave
partial column sets and chunks."""
import numpy as np
import pytest

from microfc_amd import RhsModule, ic
from oracle import oracle as O

from helpers import field_3d_case, one_fluid_3d_case, perturbed, say, stretched_grids, to_oracle

pytestmark = pytest.mark.gpu


def _stretched_2d():
    prm, _, q = ic.shock_bubble_2d(N=1237)
    prm.bc_beg, prm.bc_end = (-2, -4, -3), (-4, -2, -3)
    return prm, stretched_grids(prm), perturbed(prm, q)


CASES = {
    "stretched_2d": _stretched_2d,
    "stretched_3d": lambda: field_3d_case(126, 98, 121, (-2, -4, -1), (-4, -2, -1), grid="stretched"),
    "uniform_3d": lambda: field_3d_case(127, 127, 191, (-1, -2, -3), (-1, -2, -4)),
    "uniform_3d_one_fluid": lambda: one_fluid_3d_case(127, 127, 191, (-4, -3, -2), (-3, -2, -4)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_primitive_field_of_the_march(gpu, name):
    torch = gpu
    prm, grids, q = CASES[name]()
    oc = to_oracle(prm)
    rhs, prim = O.compute_rhs(oc, grids, q, want_prim=True)
    mod = RhsModule(prm, grids)
    try:
        say(f"[march prim] {name}")
        qd = torch.from_numpy(q.copy()).cuda()
        pd, rd = mod.new_field(), mod.new_field(ghosted=False)
        mod.timing(enable=True, reset=True)
        mod.s_compute_rhs(qd, pd, rd, 0)
        mod.sync()
        # no pass of its own for the primitive field
        assert mod.timing(enable=False)["cons_to_prim"][1] == 0
        assert np.array_equal(rd.cpu().numpy(), rhs)
        assert np.array_equal(pd.cpu().numpy(), prim)
        assert np.array_equal(qd.cpu().numpy(), O.bc_fill(oc, q.copy()))
    finally:
        mod.finalize()
