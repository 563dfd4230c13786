"""The P2P's start as the library chooses it and as the knobs say, both kept
available for a problem whose P2P outweighs its M2L."""
import numpy as np
import pytest

import datasets
import tfmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [tfmm.FP64, tfmm.MIXED])
@pytest.mark.parametrize("graph", [0, 2])
def test_gpu_choice_keeps_the_fields(precision, graph):
    """9,375 leaves of at most 64 bodies: one wave a leaf, where the library may
    choose resident waves.  Each leaf is computed the same way by either."""
    bodies = datasets.cube(600000, seed=6)
    prm = tfmm.make_params(64, 0.4, precision)
    with tfmm.Context(0) as c:
        c.set_bodies(*bodies)
        c.set_tuning(tfmm.TUNE_GRAPH, graph)
        assert c.get_tuning(tfmm.TUNE_P2P_CHOICE) == 1
        out = []
        for choice in (1, 0, 0, 1):
            print("P2P choice %d, graph %d" % (choice, graph), flush=True)
            c.set_tuning(tfmm.TUNE_P2P_CHOICE, choice)
            c.evaluate(prm)
            # another setting is another plan
            assert c.stats()["one_graph"] == (graph == 2 and len(out) == 2)
            out.append(c.fields())
            assert c.get_tuning(tfmm.TUNE_P2P_CHOICE) == choice
            assert c.get_tuning(tfmm.TUNE_P2P_SCHEDULE) == 0
        for f in out[1:]:
            assert np.array_equal(f, out[0])
        for bad in (-1, 2, 0.5):
            with pytest.raises(tfmm.TfmmError):
                c.set_tuning(tfmm.TUNE_P2P_CHOICE, bad)
