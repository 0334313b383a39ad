"""The state's way into the records with the bin's keys and counts on it, bit for
bit against the conversion alone with the bin from the records, at the edges of a
wave and of a block, in storage order and shuffled, alone and in a batch."""
import numpy as np
import pytest

from nebula_amd.mpm import MaterialModel
from nebula_amd.scenes import falling_box, make_batch_engine, make_engine

pytestmark = pytest.mark.gpu


def _scene(n, shuffled):
    rng = np.random.default_rng(n)
    sc = falling_box("a", 48, n, 2e4, 0.3, MaterialModel.VON_MISES, rng)
    sc.fields[1:, :, :3] += rng.uniform(-0.01, 0.01, (7, n, 3)).astype(np.float32)
    if shuffled:
        sc.fields[:] = sc.fields[:, rng.permutation(n)]
    return sc


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 5000])
@pytest.mark.parametrize("shuffled", [False, True])
def test_counted_conversion_equals_conversion_and_bin(gpu_lib, n, shuffled):
    sc = _scene(n, shuffled)
    a, b = make_engine(sc), make_engine(sc)
    b.runBin()                     # converts without counting
    a.substep(sc.dt, 1)
    b.substep(sc.dt, 1)
    moved = a.getState()
    assert np.array_equal(moved.view(np.uint32), b.getState().view(np.uint32))
    a.setState(sc.fields)          # counts of the last G2P are still there
    a.substep(sc.dt, 2)
    b.substep(sc.dt, 1)
    two = b.getState()
    assert np.array_equal(a.getState().view(np.uint32), two.view(np.uint32))
    c = make_batch_engine([sc, _scene(n + 3, shuffled)])
    c.substep(sc.dt, 2)
    got = c.getState()[:, :n].copy()
    got[1, :, 3] = two[1, :, 3]    # the batch's material ids are offset
    assert np.array_equal(got.view(np.uint32), two.view(np.uint32))
