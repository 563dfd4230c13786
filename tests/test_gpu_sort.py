"""The key sort around its tiles: sizes at the edges of one tile of 4,096 keys,
and around the 32 tiles up to which the scatter sums the counts by itself."""
import numpy as np
import pytest

import tfmm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = tfmm.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [1, 2, 4095, 4096, 4097, 131072, 131073, 200001])
@pytest.mark.parametrize("spread", ["uniform", "few"])
def test_gpu_key_sort(ctx, n, spread):
    """Keys ascend, equal keys keep the input's order, and the keys are those of
    the same bodies in any other order."""
    r = np.random.default_rng(n)
    x, y, z = r.random((3, n)) if spread == "uniform" else r.integers(0, 3, (3, n)) / 2.0
    q = np.ones(n)
    prm = tfmm.make_params(64, 0.4, tfmm.FP64)
    print("sort n=%d %s" % (n, spread), flush=True)
    ctx.set_bodies(x, y, z, q)
    ctx.build_tree(prm)
    keys, perm = [a.copy() for a in ctx.sorted()]
    assert np.array_equal(np.sort(perm), np.arange(n))
    assert np.all(keys[1:] >= keys[:-1])
    same = keys[1:] == keys[:-1]
    assert np.all(perm[1:][same] > perm[:-1][same])
    o = r.permutation(n)
    ctx.set_bodies(x[o], y[o], z[o], q)
    ctx.build_tree(prm)
    assert np.array_equal(ctx.sorted()[0], keys)
