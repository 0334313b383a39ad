"""P2G item by item against the box form, bit for bit: a scene on its own takes
the items up to 262,144 particles and 144 occupied tiles, the same scene in a
batch with a large one takes the boxes.  Sizes around the rule's lines (waves per
item, particles, tiles), the smallest ones, and cells crowded beyond one item and
one wave."""
import numpy as np
import pytest

from nebula_amd.mpm import MaterialModel
from nebula_amd.scenes import falling_box, make_batch_engine, make_engine

pytestmark = pytest.mark.gpu

_filler = []


def _fill():
    if not _filler:
        _filler.append(falling_box("fill", 96, 262145, 2e4, 0.3, MaterialModel.ELASTIC, np.random.default_rng(3)))
    return _filler[0]


@pytest.mark.parametrize("n,lo,size", [
    (1, 0.5, 0.01), (65, 0.4, 0.2), (4096, 0.3, 0.2), (3000, 0.45, 0.03), (900, 0.5, 0.01), (32768, 0.3, 0.35),
    (32769, 0.05, 0.9), (60000, 0.1, 0.65), (98304, 0.3, 0.4), (98305, 0.3, 0.4), (262144, 0.2, 0.5),
    (262145, 0.2, 0.5)])
@pytest.mark.parametrize("item", [4, 12, 32])
def test_items_equal_boxes(gpu_lib, n, lo, size, item):
    rng = np.random.default_rng(n + item)
    sc = falling_box("a", 64, n, 2e4, 0.3, MaterialModel.DRUCKER_PRAGER if n % 2 else MaterialModel.ELASTIC, rng)
    sc.fields[0, :, :3] = (lo + size * rng.random((n, 3))).astype(np.float32)
    sc.fields[1, :, :3] = rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32)
    one, two = make_engine(sc), make_batch_engine([sc, _fill()])
    for e in (one, two):
        t = e.tuning()
        t.p2g_item = item
        e.setTuning(t)
        e.substep(sc.dt, 3)
    a = one.getState()
    _, first, count = two.sceneInfo(0)
    b = two.getState()[:, first:first + count].copy()
    b[1, :, 3] = a[1, :, 3]  # the batch's material ids are offset
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
