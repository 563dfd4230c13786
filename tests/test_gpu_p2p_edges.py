"""The P2P where its list sort and its pair arithmetic change branch: source
lists around the sizes of the in-register sorts, and FP64 pairs at widths and
distances far from 1."""
import numpy as np
import pytest

import oracle
import tfmm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = tfmm.Context(0)
    yield c
    c.close()


def test_gpu_list_lengths(ctx):
    """One target for each length; its sources come back in order."""
    r = np.random.default_rng(5)
    n = 6000
    x, y, z = [r.random(n) for _ in range(3)]
    ctx.set_bodies(x, y, z, r.uniform(-1, 1, n))
    ctx.build_tree(tfmm.make_params(1, 0.4, tfmm.FP64))
    c = ctx.cells()
    leaves = np.flatnonzero((c["leaf"] == 1) & (c["nb"] > 0)).astype(np.int32)
    lens = [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1025]
    src = {int(t): r.choice(leaves, k, replace=False) for t, k in zip(leaves, lens)}
    p2p = np.concatenate([np.stack([np.full(len(s), t, np.int32), s], 1) for t, s in src.items()])
    r.shuffle(p2p)
    print("list lengths %s" % lens, flush=True)
    ctx.upward()
    ctx.traverse_lists(np.zeros((0, 2), np.int32), p2p)
    _, (po, ps) = ctx.lists()
    for t, s in src.items():
        assert np.array_equal(ps[po[t]:po[t + 1]], np.sort(s)), len(s)


@pytest.mark.parametrize("width", [1e-60, 1e-6, 1.0, 1e12, 1e30])
def test_gpu_fp64_pairs_at_any_width(ctx, width):
    """One leaf: the P2P alone is the field.  Coincident bodies do not interact,
    and bodies 1e-13 of the width apart do."""
    r = np.random.default_rng(9)
    n = 60
    x, y, z = [width * r.uniform(-1, 1, n) for _ in range(3)]
    q = r.random(n) + 0.5
    x[1], y[1], z[1] = x[0], y[0], z[0]
    x[2], y[2], z[2] = 0, 0, 0
    x[3], y[3], z[3] = 1e-13 * width, 0, 0
    print("one leaf of width %g" % width, flush=True)
    ctx.set_bodies(x, y, z, q)
    ctx.evaluate(tfmm.make_params(64, 0.4, tfmm.FP64))
    f, ref = ctx.fields(), oracle.direct(x, y, z, q, np.arange(n))
    # 1/r to 4.1e-15 and its cube in the acceleration, sums of 60 terms
    assert np.allclose(f[:, 0], ref[:, 0], rtol=2e-14, atol=0)
    far = np.arange(n) != 2
    assert np.all(np.linalg.norm(f - ref, axis=1)[far] <=
                  5e-14 * np.linalg.norm(np.abs(ref) + np.abs(ref).max(1, keepdims=True), axis=1)[far])


@pytest.mark.parametrize("n,ncrit", [(5, 8), (512, 1), (600, 1), (3000, 1), (9000, 1), (600, 300),
                                     (20000, 16)])
@pytest.mark.parametrize("precision,tol", [(tfmm.FP64, 1e-12), (tfmm.MIXED, 1e-6)])
def test_gpu_waves_per_leaf(ctx, n, ncrit, precision, tol):
    """Every number of waves a leaf (8, 4, 2 and 1, by n / ncrit), lists shorter
    than it, and the resident form bit for bit the same."""
    r = np.random.default_rng(n)
    x, y, z = [r.random(n) for _ in range(3)]
    q = r.random(n) + 0.5
    print("n=%d ncrit=%d precision %d" % (n, ncrit, precision), flush=True)
    ctx.set_bodies(x, y, z, q)
    prm = tfmm.make_params(ncrit, 0.5, precision)
    ctx.evaluate(prm)
    f = ctx.fields()
    ctx.set_tuning(tfmm.TUNE_P2P_WAVES, 2)
    try:
        ctx.evaluate(prm)
        assert np.array_equal(ctx.fields(), f)
    finally:
        ctx.set_tuning(tfmm.TUNE_P2P_WAVES, 0)
    # against the oracle's evaluation: FP64 differs by rounding, mixed by the
    # rounding of FP32 pairs (6e-8) and, in the far field, of FP32 M2L
    ep, ea = oracle.rel_l2(f, oracle.Run(x, y, z, q, ncrit, 0.5, phases=3).fields())
    assert ep < tol and ea < 4 * tol, (ep, ea)


@pytest.mark.parametrize("precision", [tfmm.FP64, tfmm.MIXED])
def test_gpu_chosen_p2p_start(ctx, precision):
    """Where the P2P outweighs the M2L the library starts it early by itself; the
    fields are those of a start that the caller sets, bit for bit, with and without
    the one-launch graph, and after bodies for which it chooses otherwise."""
    r = np.random.default_rng(4)
    big = [r.random(600000) for _ in range(3)] + [r.random(600000) + 0.5]
    small = [v[:3000] for v in big]
    prm = tfmm.make_params(64, 0.5, precision)
    print("chosen P2P start, precision %d" % precision, flush=True)
    ctx.set_bodies(*big)
    ctx.set_tuning(tfmm.TUNE_P2P_SCHEDULE, 1)
    try:
        ctx.evaluate(prm)
        ref = ctx.fields()
        ctx.set_tuning(tfmm.TUNE_P2P_SCHEDULE, 0)
        for graph in (0, 2):
            ctx.set_tuning(tfmm.TUNE_GRAPH, graph)
            for bodies in (big, big, small, big, big):
                ctx.set_bodies(*bodies)
                ctx.evaluate(prm)
                if bodies is big:
                    assert np.array_equal(ctx.fields(), ref), graph
    finally:
        ctx.set_tuning(tfmm.TUNE_P2P_SCHEDULE, 0)
        ctx.set_tuning(tfmm.TUNE_GRAPH, 0)
