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


def shaped(kind, n, seed):
    r = np.random.default_rng(seed)
    p = r.random((3, n))
    if kind == "cluster":  # all but two far closer together than the last bodies
        p = 0.5 + 1e-5 * p
        p[:, 0], p[:, 1] = 0, 1
    elif kind == "runs":  # groups of 100 to 600 bodies that agree to level 16
        g = r.integers(0, max(1, n // 300), n)
        p = r.random((3, n // 300 + 1))[:, g] + 2.0 ** -17 * p
    elif kind == "points":  # 700 bodies in one point
        p[:, :700] = 0.3
    return p[0], p[1], p[2], np.ones(n)


@pytest.mark.parametrize("graph", [0, 2])
def test_gpu_key_prefix_sort(graph):
    """Sorting by leading bits and runs, with the last tree's depth at hand, gives
    the order of the whole keys as a fresh context sorts them, also where runs
    cross workgroups, are too long, or the bodies draw together."""
    prm = tfmm.make_params(64, 0.6, tfmm.FP64)
    kept = tfmm.Context(0)
    kept.set_tuning(tfmm.TUNE_GRAPH, graph)
    try:
        for i, (kind, n) in enumerate([("cube", 5000), ("cube", 5000), ("runs", 5000),
                                       ("cluster", 5000), ("cluster", 5000), ("points", 5000),
                                       ("points", 5000), ("runs", 5000), ("cube", 4099),
                                       ("cube", 4099), ("cube", 60000), ("runs", 60000),
                                       ("runs", 60000)]):
            b = shaped(kind, n, i)
            print("prefix sort %d: %s n=%d graph %d" % (i, kind, n, graph), flush=True)
            kept.set_bodies(*b)
            kept.evaluate(prm)
            keys, perm = [a.copy() for a in kept.sorted()]
            fresh = tfmm.Context(0)
            try:
                fresh.set_bodies(*b)
                fresh.build_tree(prm)
                fk, fp = fresh.sorted()
                assert np.array_equal(keys, fk) and np.array_equal(perm, fp), (i, kind)
            finally:
                fresh.close()
    finally:
        kept.close()


def test_gpu_key_prefix_sort_batch():
    """The same in a forest: runs end at the problems' ends."""
    prm = tfmm.make_params(16, 0.6, tfmm.FP64)
    kept = tfmm.Context(0)
    try:
        for i, kinds in enumerate([["cube"] * 9, ["cube"] * 9, ["runs"] * 9, ["cluster"] * 9,
                                   ["cube", "runs", "cluster"] * 3]):
            probs = [shaped(k, 901 + 40 * j, 10 * i + j) for j, k in enumerate(kinds)]
            print("prefix sort of a batch, %s" % kinds[:3], flush=True)
            kept.set_batch(probs)
            kept.evaluate(prm)
            keys, perm = [a.copy() for a in kept.sorted()]
            fresh = tfmm.Context(0)
            try:
                fresh.set_batch(probs)
                fresh.build_tree(prm)
                fk, fp = fresh.sorted()
                assert np.array_equal(keys, fk) and np.array_equal(perm, fp), i
            finally:
                fresh.close()
    finally:
        kept.close()
