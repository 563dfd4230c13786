"""M2L pairs outside the offset groups: a plan made from an evaluation without any
has no place for them, so bodies that bring some run the ordinary way and leave a
plan that has; with periodic images their keys hold the whole source word."""
import numpy as np
import pytest

import datasets
import oracle
import tfmm

pytestmark = pytest.mark.gpu


def test_gpu_plan_without_outside_pairs():
    prm = tfmm.make_params(16, 0.4, tfmm.FP64)
    none, some = datasets.cube(20000, seed=4), datasets.two_plummer(20000, seed=3)
    ref, ctx = tfmm.Context(0), tfmm.Context(0)
    try:
        want = []
        for b in (none, some):
            ref.set_bodies(*b)
            ref.evaluate(prm)
            want.append((ref.fields(), ref.stats()["n_m2l_fallback"]))
        assert want[0][1] == 0 and want[1][1] > 0
        ctx.set_tuning(tfmm.TUNE_GRAPH, 2)
        for rep, which in enumerate((0, 0, 1, 1, 1, 0, 0)):
            print("evaluation %d, outside pairs: %d" % (rep, want[which][1]), flush=True)
            ctx.set_bodies(*(none, some)[which])
            ctx.evaluate(prm)
            assert np.array_equal(ctx.fields(), want[which][0]), rep
            assert ctx.stats()["n_m2l_fallback"] == want[which][1]
    finally:
        ref.close()
        ctx.close()


@pytest.mark.parametrize("images", [1, 2])
def test_gpu_periodic_outside_pairs(images):
    """FP64 within relative L2 1e-10 of the CPU oracle."""
    rng = np.random.default_rng(9)
    n, half = 6000, np.pi
    # half of the bodies in a ball beside a face, the others everywhere
    ball = rng.normal(scale=0.004, size=(n // 2, 3)) + [half - 0.1, 0.2, -0.3]
    pos = np.concatenate([ball, rng.uniform(-half, half, size=(n - n // 2, 3))])
    x, y, z = (np.ascontiguousarray(v) for v in pos.T)
    q = rng.uniform(-1, 1, size=n)
    c = tfmm.Context(0)
    try:
        c.set_periodic(images, 2 * half)
        c.set_bodies(x, y, z, q)
        c.evaluate(tfmm.make_params(8, 0.4, tfmm.FP64))
        assert c.stats()["n_m2l_fallback"] > 0
        o = oracle.Run(x, y, z, q, 8, 0.4, images=images, cycle=2 * half)
        ep, ea = oracle.rel_l2(c.fields(), o.fields())
        print("images %d: %d pairs outside, %.2e %.2e" % (
            images, c.stats()["n_m2l_fallback"], ep, ea))
        assert ep < 1e-10 and ea < 1e-10
    finally:
        c.close()
