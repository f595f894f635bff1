"""The CFL reduction where its blocks change: one cell less than a block's
chunk of 1024 cells, a whole chunk, one more; one block for each of its 512,
one cell more (a second chunk); the maximum in the first and in the last cell.
Bitwise the oracle's maximum, on repeated calls, and a NaN anywhere is kept."""
import numpy as np
import pytest

from microfc_amd import RhsModule, ic
from oracle import oracle as O

from helpers import say, to_oracle


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [25, 1023, 1024, 1025, 512 * 1024, 512 * 1024 + 1])
def test_icfl_at_the_edges_of_blocks(gpu, cells):
    torch = gpu
    prm, grids, q = ic.sod_1d(m=cells - 1)
    oc = to_oracle(prm)
    b = (q.shape[-1] - cells) // 2
    mod = RhsModule(prm, grids)
    try:
        for at in (0, cells // 2, cells - 1):
            say(f"[cfl blocks] {cells} cells, maximum in cell {at}")
            prim = O.cons_to_prim(oc, q)
            prim[prm.num_fluids, ..., b + at] = 50.0  # the velocity
            qd = torch.from_numpy(prim).cuda()
            want = O.icfl_max(oc, grids, prim, 1e-6)
            for _ in range(2):
                assert mod.icfl_max(qd, 1e-6) == want
            prim[prm.num_fluids, ..., b + at] = np.nan
            assert np.isnan(mod.icfl_max(torch.from_numpy(prim).cuda(), 1e-6))
            assert mod.icfl_max(qd, 1e-6) == want
    finally:
        mod.finalize()
