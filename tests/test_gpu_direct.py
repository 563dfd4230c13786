"""The FP64 direct sum where its split of the targets and bodies changes:
target counts around the lines between 1, 2 and 4 targets a workgroup, body
counts around a workgroup's threads, repeated targets, coincident bodies, and
periodic images, against the oracle."""
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


@pytest.mark.parametrize("n", [1, 511, 513, 1500])
@pytest.mark.parametrize("nt", [1, 1023, 1025, 2049])
@pytest.mark.parametrize("images", [0, 1])
def test_gpu_direct_splits(ctx, n, nt, images):
    r = np.random.default_rng(n + nt)
    x, y, z = [r.uniform(-1, 1, n) for _ in range(3)]
    q = r.random(n) + 0.5
    if n > 2:
        x[1], y[1], z[1] = x[0], y[0], z[0]  # no interaction between the two
    t = r.integers(0, n, nt)
    print("direct n=%d targets=%d images=%d" % (n, nt, images), flush=True)
    ctx.set_periodic(images, 2.0)
    try:
        ctx.set_bodies(x, y, z, q)
        got = ctx.direct(t)
        assert np.array_equal(got, ctx.direct_noalloc(t))
        assert np.array_equal(got[:1], ctx.direct(t[:1]))  # whatever the other targets are
    finally:
        ctx.set_periodic(0, 0.0)
    ref = (oracle.direct_periodic(x, y, z, q, t, images, 2.0) if images
           else oracle.direct(x, y, z, q, t))
    # a pair is good to a few ulp, a sum of up to 40,000 positive terms in another
    # order to 40,000 ulp at the very most, 200 as a random walk; the
    # accelerations of a symmetric set of images cancel to a tenth or less
    assert np.allclose(got[:, 0], ref[:, 0], rtol=1e-12, atol=0)
    scale = np.abs(ref[:, 1:]).max() + np.abs(ref[:, :1]).max()
    assert np.abs(got[:, 1:] - ref[:, 1:]).max() <= 1e-12 * scale
