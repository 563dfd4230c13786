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
    """32,768 leaves of 32 bodies: one wave a leaf, and more P2P than M2L, where the
    library chooses resident waves.  Each leaf is computed the same way by either."""
    bodies = datasets.cube(1 << 20, seed=6)
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
            # as the P2P ran, which bench.py names its kernel by
            mine = 3 if precision == tfmm.MIXED else 2
            assert c.p2p_start() == ((2, mine) if choice else (0, 0))
            out.append(c.fields())
            assert c.get_tuning(tfmm.TUNE_P2P_CHOICE) == choice
            assert c.get_tuning(tfmm.TUNE_P2P_SCHEDULE) == 0
        for f in out[1:]:
            assert np.array_equal(f, out[0])
        for bad in (-1, 2, 0.5):
            with pytest.raises(tfmm.TfmmError):
                c.set_tuning(tfmm.TUNE_P2P_CHOICE, bad)


def test_gpu_start_as_set():
    with tfmm.Context(0) as c:
        c.set_bodies(*datasets.cube(20000, seed=6))
        with pytest.raises(tfmm.TfmmError):
            c.p2p_start()  # nothing evaluated yet
        for schedule, waves in ((0, 0), (1, 0), (2, 3), (3, 2), (4, 0)):
            c.set_tuning(tfmm.TUNE_P2P_SCHEDULE, schedule)
            c.set_tuning(tfmm.TUNE_P2P_WAVES, waves)
            c.evaluate(tfmm.make_params(64, 0.4, tfmm.MIXED))
            # (20,000 bodies: several waves a leaf, nothing for the library to choose)
            assert c.p2p_start() == (schedule, waves)
