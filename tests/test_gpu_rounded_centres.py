"""Cells as narrow as the last place of their bodies' coordinates: the centres of
neighbouring cells round to one point, so a target meets two sources at one offset."""
import numpy as np
import pytest

import oracle
import tfmm

pytestmark = pytest.mark.gpu


def _lattice(n=20000):
    """Whole numbers 2^52 + 0 ... 15, where the next number is 1 away, and a corner
    that makes the box 16 wide: the cells of level 4 have width 1."""
    r = np.random.default_rng(1)
    x, y, z = [2.0 ** 52 + r.integers(0, 16, n).astype(float) for _ in range(3)]
    x[-1] = y[-1] = z[-1] = 2.0 ** 52 + 16
    x[-2] = y[-2] = z[-2] = 2.0 ** 52
    return x, y, z, r.uniform(-1, 1, n)


@pytest.mark.parametrize("precision", [tfmm.FP64, tfmm.MIXED])
def test_gpu_centres_that_round_together(precision):
    x, y, z, q = _lattice()
    n_m2l = oracle.Run(x, y, z, q, 20, 0.5).counts()["m2l"]
    # FP64; FP32 operands in mixed precision
    tol = 1e-12 if precision == tfmm.FP64 else 1e-5
    prm = tfmm.make_params(20, 0.5, precision)

    def counted(c):
        st = c.stats()
        assert st["n_m2l"] == n_m2l
        # 76,174 pairs have no place in the groups, 37,156 repeat one
        assert st["n_m2l_fallback"] == 76174 + 37156

    with tfmm.Context(0) as c:
        c.set_bodies(x, y, z, q)
        print("rounded centres, the stages' calls", flush=True)
        c.build_tree(prm)
        c.upward()
        c.traverse()
        counted(c)
        M, L = c.expansions()
        (off, src), _ = c.lists()
        centre, nb = c.cells()["center"], c.cells()["nb"]
        for t in np.flatnonzero((np.diff(off) > 0) & (nb > 0))[::97]:
            want = np.zeros_like(M[0])
            for s in src[off[t]:off[t + 1]]:  # every pair of the list, once
                want = oracle.m2l(M[s], centre[t] - centre[s], want)
            assert np.linalg.norm(L[t] - want) < tol * np.linalg.norm(want), t
        pots = []
        for graph in (0, 2, 2, 2):
            print("rounded centres, evaluations, graph %d" % graph, flush=True)
            c.set_tuning(tfmm.TUNE_GRAPH, graph)
            c.evaluate(prm)
            counted(c)
            pots.append(c.fields()[:, 0])
        for p in pots[1:]:
            assert np.linalg.norm(p - pots[0]) < tol * np.linalg.norm(pots[0])
