"""The reductions over the cells (mfc_cfl_dt, mfc_cfl_dt_noalloc, mfc_icfl_max,
mfc_stability_criteria) called from several host threads at once, on fields
whose values differ: each call returns its own field's value, bit for bit the
one it returns alone.  They share a block counter and a result word, so a call
that overlapped another would take the other's."""
import ctypes
import threading

import pytest

from microfc_amd import RhsModule, ic

from helpers import say

pytestmark = pytest.mark.gpu


def test_reductions_from_several_threads(gpu):
    torch = gpu
    prm, grids, q = ic.viscous_shear_2d(N=256)
    mod = RhsModule(prm, grids)
    try:
        lib, S = mod.lib, prm.sys_size
        cons, prims = [], []
        for k in range(4):
            qd = torch.from_numpy(q.copy()).cuda()
            qd[prm.num_fluids:prm.num_fluids + 2] *= 1.0 - 0.2 * k  # the momenta (the pressure rises)
            pd = mod.new_field()
            mod.s_convert_conservative_to_primitive_variables(qd, pd)
            cons.append(qd)
            prims.append(pd)
        mod.sync()
        cp, pp = [mod._ptrs(t) for t in cons], [mod._ptrs(t) for t in prims]

        def call(kind, k):
            out = (ctypes.c_double * 3)()
            at = ctypes.cast(out, ctypes.POINTER(ctypes.c_double))
            if kind == 0:
                rc = lib.mfc_cfl_dt(cp[k], 0.4, at)
            elif kind == 1:
                rc = lib.mfc_cfl_dt_noalloc(cp[k], 0.4, at)
            elif kind == 2:
                rc = lib.mfc_icfl_max(pp[k], 1e-6, at)
            else:
                rc = lib.mfc_stability_criteria(pp[k], 1e-6, out)
            return rc, tuple(out)

        want = {(kind, k): call(kind, k) for kind in range(4) for k in range(4)}
        assert all(rc == 0 for rc, _ in want.values())
        assert len({want[0, k][1] for k in range(4)}) == 4
        wrong = []

        def work(kind, k):
            for r in range(200):
                at = (kind, (k + r) % 4)
                got = call(*at)
                if got != want[at]:
                    wrong.append((at, got, want[at]))

        for kinds in ((0, 1), (0, 1, 2, 3), (1, 1, 0, 0)):
            ts = [threading.Thread(target=work, args=(kind, i)) for i, kind in enumerate(kinds)]
            for t in ts:
                t.start()
            for t in ts:
                t.join()
            say(f"[cfl threads] kinds {kinds}: {len(wrong)} wrong")
            assert not wrong, wrong[:3]
    finally:
        mod.finalize()
