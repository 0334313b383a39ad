"""What a call can read after a graph replay (nb_mpm_graph_substeps): bins and
grid must be those of its last substep, as after eager substeps, also when the
replay uses an earlier capture and the state, the grid or the bins were replaced
in between."""
import numpy as np
import pytest

from nebula_amd.scenes import make_engine
from test_gpu_batch import _scenes

pytestmark = pytest.mark.gpu


def _between(name, e, sc):
    """Something other than a substep between two replays; the state is rewritten."""
    st = e.getState()
    if name == "recorded run":
        e.adjointBegin(4, 2)
        e.forwardRecorded(sc.dt)
        e.setAdjoint(np.ones_like(st))
        e.backward()
        e.adjointEnd()
    elif name == "grid written":
        mom, mass = e.getGrid()
        e.setGrid(mom + 1.0, mass + 1.0)
    elif name == "fused":
        e.setFusedG2P(True)
        e.substep(sc.dt, 2)
        e.setFusedG2P(False)
    st[1, :, :3] *= 0.5
    e.setState(st)


@pytest.mark.parametrize("name, flip_ratio", [("state written", -1.0), ("state written", 0.95), ("recorded run", -1.0),
                                              ("grid written", -1.0), ("grid written", 0.95), ("fused", -1.0),
                                              ("fused", 0.95)])
def test_bins_and_grid_after_a_replay(gpu_lib, name, flip_ratio):
    sc = _scenes(flip_ratio=flip_ratio, corrected=True)[1]
    eager, graph = make_engine(sc), make_engine(sc)
    eager.substep(sc.dt, 3)
    graph.graphSubstep(sc.dt, 3)
    for e in (eager, graph):
        _between(name, e, sc)
    eager.substep(sc.dt, 3)
    graph.graphSubstep(sc.dt, 3)
    for what, a, b in zip(("momentum", "mass"), eager.getGrid(), graph.getGrid()):
        assert np.any(a), what
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), what
    for what, a, b in zip(("keys", "sorted", "count", "end"), eager.getBins(), graph.getBins()):
        assert np.array_equal(a, b), what
    assert np.array_equal(eager.getState().view(np.uint32), graph.getState().view(np.uint32))


@pytest.mark.parametrize("n", [1, 2, 5])
def test_fallback_queue_is_worked_off_within_the_call(gpu_lib, n):
    """Every particle takes the FP64 fallback (equal singular values): a replayed run's
    last queue is settled with that run's time step, and nothing of it is left for the
    standalone G2P, whose own entries need the whole queue."""
    sc = _scenes()[2]
    sc.fields[2:5, :, :3] = (np.eye(3) * (0.98, 0.95, 0.98))[:, None]
    eager, graph = make_engine(sc), make_engine(sc)
    for e, run in ((eager, eager.substep), (graph, graph.graphSubstep)):
        e.setSvdFallback(count_stats=True)
        e.svdFallbackStats(reset=True)
        for dt in (sc.dt, 0.5 * sc.dt):
            run(dt, n)
            e.runBin()
            e.runG2P(dt)
    assert eager.svdFallbackStats() == graph.svdFallbackStats()
    assert eager.svdFallbackStats()["fp64_return_map_lanes"] >= sc.n
    assert np.array_equal(eager.getState().view(np.uint32), graph.getState().view(np.uint32))
