"""The tree's first levels in one workgroup (built with the last tree's level
sizes at hand) against the tree of a fresh context (built level by level), as
the levels grow, shrink and change shape between the trees, and with more roots
than the workgroup has threads."""
import numpy as np
import pytest

import datasets
import tfmm

pytestmark = pytest.mark.gpu


def cells(ctx, prm):
    ctx.build_tree(prm)
    return {k: np.array(v) for k, v in ctx.cells().items()}


def same(a, b):
    assert a.keys() == b.keys()
    for k in a:
        assert np.array_equal(a[k], b[k]), k


def test_gpu_tree_follows_earlier_shapes():
    steps = [(datasets.cube(3000, seed=1), 8), (datasets.cube(3000, seed=1), 8),
             (datasets.plummer(3000, seed=2), 8), (datasets.cube(40000, seed=3), 4),
             (datasets.cube(40000, seed=4), 4), (datasets.ellipsoid(70, seed=5), 64),
             (datasets.cube(1, seed=6), 1), (datasets.plummer(20000, seed=7), 1),
             (datasets.plummer(20000, seed=7), 1)]
    kept = tfmm.Context(0)
    try:
        for i, (b, ncrit) in enumerate(steps):
            print("tree %d: n=%d ncrit=%d" % (i, len(b[0]), ncrit), flush=True)
            prm = tfmm.make_params(ncrit, 0.5, tfmm.FP64)
            kept.set_bodies(*b)
            got = cells(kept, prm)
            fresh = tfmm.Context(0)
            try:
                fresh.set_bodies(*b)
                same(got, cells(fresh, prm))
            finally:
                fresh.close()
    finally:
        kept.close()


@pytest.mark.parametrize("problems", [3, 1025])
def test_gpu_forest_tree_twice(problems):
    probs = [datasets.cube(20 + 3 * (i % 5), seed=i) for i in range(problems)]
    print("forest of %d" % problems, flush=True)
    ctx = tfmm.Context(0)
    try:
        ctx.set_batch(probs)
        prm = tfmm.make_params(4, 0.5, tfmm.FP64)
        first = cells(ctx, prm)
        same(cells(ctx, prm), first)
    finally:
        ctx.close()
