"""The phase times of tfmm_stats_t: each part of an evaluation in one phase."""
import numpy as np
import pytest

import datasets
import tfmm

pytestmark = pytest.mark.gpu

PHASES = ("ms_tree", "ms_upward", "ms_traverse", "ms_downward")


def _times(c, prm, reps=7):
    c.evaluate(prm)
    c.evaluate(prm)
    st = []
    for _ in range(reps):
        c.evaluate(prm)
        st.append(c.stats())
    return {k: float(np.median([s[k] for s in st])) for k in PHASES + ("ms_total", "ms_m2l")}, st


@pytest.mark.parametrize("graph", [0, 1, 2])
@pytest.mark.parametrize("schedule,waves", [(0, 0), (0, 3), (1, 0), (2, 3), (3, 2), (4, 0)])
def test_gpu_phases_add_up(graph, schedule, waves):
    """The upward pass on the context stream (schedules 2 to 4, and a numeric phase
    that is a graph): the phases follow one another.  Otherwise it runs beside the
    traversal, and the others do."""
    with tfmm.Context(0) as c:
        c.set_bodies(*datasets.plummer(100000, seed=8, charges="uniform"))
        c.set_tuning(tfmm.TUNE_GRAPH, graph)
        c.set_tuning(tfmm.TUNE_P2P_CHOICE, 0)
        c.set_tuning(tfmm.TUNE_P2P_SCHEDULE, schedule)
        c.set_tuning(tfmm.TUNE_P2P_WAVES, waves)
        print("phase times, schedule %d waves %d graph %d" % (schedule, waves, graph), flush=True)
        _, st = _times(c, tfmm.make_params(16, 0.4, tfmm.FP64))
        for s in st:
            serial = graph == 1 or schedule >= 2
            parts = [s[k] for k in PHASES if serial or k != "ms_upward"]
            assert min(parts) > 0 and s["ms_upward"] > 0, s
            # event times have a step of 10 ns
            assert sum(parts) <= s["ms_total"] + 1e-3, (parts, s["ms_total"])


@pytest.mark.parametrize("graph", [0, 2])
def test_gpu_downward_holds_the_l2l(graph):
    """A tree of many cells and few bodies a leaf: with nothing beside it, the
    downward phase takes about as long as the separate tfmm_downward, most of it L2L."""
    prm = tfmm.make_params(4, 0.4, tfmm.FP64)
    with tfmm.Context(0) as c:
        c.set_bodies(*datasets.cube(100000, seed=8))
        ref = []
        for _ in range(5):
            c.build_tree(prm)
            c.upward()
            c.traverse()
            c.downward()
            ref.append(c.stats()["ms_downward"])
        c.set_tuning(tfmm.TUNE_GRAPH, graph)
        c.set_tuning(tfmm.TUNE_P2P_SCHEDULE, 4)
        t, _ = _times(c, prm)
        print("downward %.3f ms, %.3f in the separate call" % (t["ms_downward"], np.median(ref)),
              flush=True)
        assert t["ms_downward"] > 0.6 * np.median(ref)
