"""The M2L over target sets: the groups of mirrored offsets (on the CPU), and
on the GPU the sizes where sets, items and work units end unevenly and lists
that hold a target's offset more than once."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import datasets
import oracle
import tfmm

HERE = os.path.dirname(os.path.abspath(__file__))


def test_mirrored_groups_match_oracle(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    oracle.lib()
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe,
                    os.path.join(HERE, "native", "m2l_mirror_check.cpp"), oracle.LIB_PATH,
                    "-Wl,-rpath," + os.path.dirname(oracle.LIB_PATH)], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    assert int(out[1]) == 23 ** 3 + 6 * 24 ** 3
    # the same sums in FP64 with signs moved: acos/atan2 round differently
    assert float(out[3]) < 1e-13, out


@pytest.fixture(scope="module")
def ctx():
    c = tfmm.Context(0)
    yield c
    c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,ncrit", [(9, 1), (65, 8), (1000, 4), (5000, 1), (5003, 64)])
@pytest.mark.parametrize("unit", [0.0, 0.05])
def test_gpu_sets_match_oracle(ctx, n, ncrit, unit):
    """Few sets and a last set that is not full; units of one item and more."""
    x, y, z, q = datasets.plummer(n, seed=n, charges="uniform")
    print("plummer n=%d ncrit=%d unit=%g" % (n, ncrit, unit), flush=True)
    ctx.set_bodies(x, y, z, q)
    ctx.set_tuning(tfmm.TUNE_M2L_UNIT, unit)
    try:
        ctx.evaluate(tfmm.make_params(ncrit, 0.5, tfmm.FP64))
    finally:
        ctx.set_tuning(tfmm.TUNE_M2L_UNIT, 0)
    ep, ea = oracle.rel_l2(ctx.fields(), oracle.Run(x, y, z, q, ncrit, 0.5, phases=3).fields())
    # FP64, a few thousand terms a body in another order
    assert ep < 1e-12 and ea < 1e-12, (ep, ea)


@pytest.mark.gpu
@pytest.mark.parametrize("copies", [2, 3])
def test_gpu_repeated_list_entries(ctx, copies):
    """A given list with every pair several times, and one pair 200 times,
    adds every entry (M2L is linear in the list)."""
    x, y, z, q = datasets.cube(6000, seed=3)
    ctx.set_bodies(x, y, z, q)
    ctx.build_tree(tfmm.make_params(16, 0.5, tfmm.FP64))
    ctx.upward()
    ctx.traverse()
    (mo, ms), _ = ctx.lists()
    once = np.stack([np.repeat(np.arange(len(mo) - 1, dtype=np.int32), np.diff(mo)), ms], 1)
    nop2p = np.zeros((0, 2), np.int32)

    def local(pairs):
        ctx.build_tree(tfmm.make_params(16, 0.5, tfmm.FP64))
        ctx.upward()
        ctx.traverse_lists(np.ascontiguousarray(pairs, np.int32), nop2p)
        return ctx.expansions()[1].copy(), ctx.stats()

    print("repeated entries: %d pairs, %d copies" % (len(once), copies), flush=True)
    a, sa = local(once)
    b, sb = local(np.concatenate([once] * copies))
    c, _ = local(np.concatenate([once, np.repeat(once[:1], 200, 0)]))
    d, _ = local(once[:1])
    assert sa["n_m2l_fallback"] == 0
    assert sb["n_m2l_fallback"] == (copies - 1) * len(once)

    def rel(u, v):
        return np.linalg.norm(u - v) / np.linalg.norm(v)
    # FP64: the per-pair kernel and the set kernel differ by rounding
    assert rel(b, copies * a) < 1e-12
    assert rel(c, a + 200 * d) < 1e-12
