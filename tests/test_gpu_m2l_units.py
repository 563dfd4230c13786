"""M2L sets that really are cut into several work units, the shortest (8 items)
against one unit a set."""
import numpy as np
import pytest

import datasets
import oracle
import tfmm

pytestmark = pytest.mark.gpu


# FP64: a few thousand terms a body in another order; FP32 sums of an item, added in
# another order
@pytest.mark.parametrize("precision,tol", [(tfmm.FP64, 1e-12), (tfmm.MIXED, 1e-6)])
@pytest.mark.parametrize("n,ncrit", [(5003, 1), (20011, 4)])
def test_gpu_several_units_a_set(precision, tol, n, ncrit):
    x, y, z, q = datasets.plummer(n, seed=n, charges="uniform")
    prm = tfmm.make_params(ncrit, 0.5, precision)
    with tfmm.Context(0) as c:
        c.set_bodies(x, y, z, q)
        out = []
        for unit in (0.05, 1e6):
            print("plummer n=%d ncrit=%d unit=%g" % (n, ncrit, unit), flush=True)
            c.set_tuning(tfmm.TUNE_M2L_UNIT, unit)
            c.evaluate(prm)
            out.append(c.fields())
        st = c.stats()
        sets = (st["ncells"] + 15) // 16
        # more than two units of 8 items a set on average, and a twentieth of the mean
        # is fewer than 8
        assert 16 * sets < st["n_m2l_items"] < 160 * sets, (sets, st["n_m2l_items"])
        ep, ea = oracle.rel_l2(out[0], out[1])
        assert ep < tol and ea < tol, (ep, ea)
