"""The adjoint's scatter cell by cell against the box form, bit for bit: a scene
on its own takes the cells up to 262,144 particles and 256 occupied tiles, the
same scene in a batch with a large one takes the boxes.  Sizes around the rule's
lines (waves per cell, particles, tiles), the smallest ones, crowded cells, and
particles on stencil nodes of vanishing weight (the weight cut)."""
import numpy as np
import pytest

from nebula_amd.mpm import MaterialModel
from nebula_amd.scenes import falling_box, make_batch_engine, make_engine

pytestmark = pytest.mark.gpu

_filler = []


def _fill():
    if not _filler:
        _filler.append(falling_box("fill", 64, 262145, 2e4, 0.3, MaterialModel.ELASTIC, np.random.default_rng(3),
                                   corrected_svd=True))
    return _filler[0]


def _gradient(e, sc, W, part=slice(None)):
    e.adjointBegin(3, 2)
    e.forwardRecorded(sc.dt)
    e.setAdjoint(W)
    e.backward()
    g = e.getAdjoint()[:, part].copy()
    e.adjointEnd()
    return g


@pytest.mark.parametrize("n,lo,size,cut", [
    (1, 0.5, 0.01, False), (65, 0.4, 0.2, True), (900, 0.5, 0.01, False), (3000, 0.45, 0.03, True),
    (32768, 0.3, 0.35, True), (60000, 0.06, 0.88, False), (131072, 0.3, 0.4, False), (131073, 0.25, 0.5, True),
    (262144, 0.2, 0.5, False), (262145, 0.2, 0.5, False)])
def test_cells_equal_boxes(gpu_lib, n, lo, size, cut):
    rng = np.random.default_rng(n)
    sc = falling_box("a", 64, n, 2e4, 0.3, MaterialModel.DRUCKER_PRAGER if n % 2 else MaterialModel.ELASTIC, rng,
                     corrected_svd=True)
    x = (lo + size * rng.random((n, 3))).astype(np.float32)
    if cut:  # a few on a cell face in three axes, a rounding away from it: weights near zero
        m = rng.random(n) < 0.05
        x[m] = (np.floor(x[m] * 64) / 64 + 1e-7).astype(np.float32)
    sc.fields[0, :, :3] = x
    sc.fields[1, :, :3] = rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32)
    W = rng.standard_normal((8, n, 4)).astype(np.float32)
    W[1, :, 3] = 0.0
    fill = _fill()
    a = _gradient(make_engine(sc), sc, W)
    b = _gradient(make_batch_engine([sc, fill]), sc, np.concatenate([W, np.zeros((8, fill.n, 4), np.float32)], axis=1),
                  slice(0, n))
    assert np.isfinite(a).all()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
