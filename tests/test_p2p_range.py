"""The FP64 P2P over the whole range of distances and charges: the rule for its
scaled coordinates (on the CPU), and on the GPU bodies outside the box that sets
the cells' widths, pairs far closer than a cell and charges far from 1."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import datasets
import oracle
import tfmm

HERE = os.path.dirname(os.path.abspath(__file__))


def test_scale_keeps_pairs_in_range(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe,
                    os.path.join(HERE, "native", "p2p_range_check.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    scaled, wide = int(out.stdout.split()[1]), int(out.stdout.split()[3])
    assert scaled > 1000 and wide > 1000


@pytest.fixture(scope="module")
def ctx():
    c = tfmm.Context(0)
    yield c
    c.close()


def _outside(width, n=40):
    """Body 0 at (1, 0, 0), the others around the origin: the box, which leaves out
    body 0's x and y, is `width` wide.  Two bodies: body 1 at the origin."""
    if width == 0:
        return np.array([1.0, 0]), np.zeros(2), np.zeros(2), np.ones(2)
    r = np.random.default_rng(3)
    x, y, z = [width * r.uniform(-0.5, 0.5, n) for _ in range(3)]
    x[0], y[0] = 1.0, 0.0
    return x, y, z, r.random(n) + 0.5


def _close(gap, n=40):
    """Bodies of a unit box, three of them `gap` apart at the origin."""
    r = np.random.default_rng(4)
    x, y, z = [r.uniform(-0.5, 0.5, n) for _ in range(3)]
    x[1:4], y[1:4], z[1:4] = [0, gap, 0], [0, 0, gap], 0
    return x, y, z, r.random(n) + 0.5


def _charges(scale, n=40):
    x, y, z, q = _close(1e-3, n)
    return x, y, z, q * scale


CASES = {"zero width": lambda: _outside(0), "width 1e-20": lambda: _outside(1e-20),
         "width 1e-30": lambda: _outside(1e-30), "width 1e-60": lambda: _outside(1e-60),
         "gap 1e-70": lambda: _close(1e-70), "gap 1e-90": lambda: _close(1e-90),
         "gap 1e-100": lambda: _close(1e-100), "charges 1e-140": lambda: _charges(1e-140),
         "charges 1e140": lambda: _charges(1e140)}


def _check(f, bodies):
    """One leaf: the P2P alone is the field.  1/r to 4.1e-15, its cube in the
    acceleration, sums of 40 terms.  (A body at the leaf's centre has no
    acceleration in the reference: its local expansion divides by the distance.)"""
    ref = oracle.direct(*bodies, np.arange(len(bodies[0])))
    assert np.allclose(f[:, 0], ref[:, 0], rtol=2e-14, atol=0)
    ok = np.all(np.isfinite(f), 1)
    assert ok[0] and ok.sum() >= len(ok) - 1
    a, b = f[ok, 1:], ref[ok, 1:]
    assert np.all(np.abs(a - b) <= 1e-13 * np.abs(b).max(1, keepdims=True))


@pytest.mark.gpu
@pytest.mark.parametrize("waves", [0, 2])
@pytest.mark.parametrize("case", CASES)
def test_gpu_fp64_range(ctx, case, waves):
    bodies = CASES[case]()
    print("FP64 P2P, %s, %d resident waves" % (case, waves), flush=True)
    ctx.set_bodies(*bodies)
    ctx.set_tuning(tfmm.TUNE_P2P_WAVES, waves)
    try:
        ctx.evaluate(tfmm.make_params(64, 0.4, tfmm.FP64))
    finally:
        ctx.set_tuning(tfmm.TUNE_P2P_WAVES, 0)
    _check(ctx.fields(), bodies)


@pytest.mark.gpu
def test_gpu_fp64_range_in_a_forest_and_a_graph(ctx):
    """Beside ordinary problems, and as one graph launch recorded for ordinary
    bodies: the same rule over all problems of an evaluation."""
    odd = [CASES[k]() for k in ("zero width", "width 1e-30", "gap 1e-90")]
    cube = datasets.cube(3000, seed=5)
    prm = tfmm.make_params(64, 0.4, tfmm.FP64)
    print("a forest with a problem of zero width", flush=True)
    ctx.set_batch([odd[0], cube, odd[1], odd[2]])
    ctx.evaluate(prm)
    f, off = ctx.fields(), ctx.problem_offsets()
    for p, b in zip((0, 2, 3), odd):
        _check(f[off[p]:off[p + 1]], b)
    ref = oracle.Run(*cube, 64, 0.4).fields()
    ep, ea = oracle.rel_l2(f[off[1]:off[2]], ref)
    assert ep < 1e-12 and ea < 1e-12, (ep, ea)
    print("a graph recorded for a unit box", flush=True)
    ctx.set_tuning(tfmm.TUNE_GRAPH, 2)
    try:
        for b in (_close(1e-3), _close(1e-3), _close(1e-90), _outside(1e-30), _close(1e-3)):
            ctx.set_bodies(*b)
            ctx.evaluate(prm)
            _check(ctx.fields(), b)
    finally:
        ctx.set_tuning(tfmm.TUNE_GRAPH, 0)


@pytest.mark.gpu
def test_gpu_mixed_zero_width(ctx):
    bodies = _outside(0)
    ctx.set_bodies(*bodies)
    ctx.evaluate(tfmm.make_params(64, 0.4, tfmm.MIXED))
    f, ref = ctx.fields(), oracle.direct(*bodies, np.arange(2))
    # a pair in FP32
    assert np.allclose(f[:, 0], ref[:, 0], rtol=1e-6) and np.allclose(f[0], ref[0], rtol=1e-6)
