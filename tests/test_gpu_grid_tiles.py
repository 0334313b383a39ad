"""The grid update per occupied tile against the form per node tile (taken with a
noise force in the list, here of strength zero), and with a tile's own and outer
nodes in one block (more than 512 tiles) against two: lone tiles, corners and walls
of the cube, a cube of one tile, neighbours in every direction.  Values equal; the
backward likewise."""
import numpy as np
import pytest

from nebula_amd import mpm
from nebula_amd.mpm import MaterialModel
from nebula_amd.scenes import falling_box, make_batch_engine, make_engine

pytestmark = pytest.mark.gpu

NOISE0 = mpm.NoiseForce((0.0, 1.0, 0.0), 0.0, 1.3, 2, 0.7, 0.1)


def _scene(grid, n, where):
    rng = np.random.default_rng(grid + n)
    sc = falling_box("a", grid, n, 2e4, 0.3, MaterialModel.ELASTIC, rng, corrected_svd=True)
    size = grid / 64.0
    u = rng.random((n, 3))
    if where == "corners":
        u = np.where(rng.random((n, 3)) < 0.5, 0.2 * u, 1.0 - 0.2 * u)
    elif where == "faces":  # along the faces between tiles
        u = (np.round(u * grid / 8) * 8 + rng.uniform(-1.2, 1.2, (n, 3))) / grid
    sc.fields[0, :, :3] = np.clip(u * size, 1e-3, size - 1e-3).astype(np.float32)
    sc.fields[1, :, :3] = rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32)
    sc.forces = []
    return sc


@pytest.mark.parametrize("where", ["anywhere", "corners", "faces"])
@pytest.mark.parametrize("grid,n", [(8, 40), (20, 1), (24, 500), (64, 7), (64, 400), (61, 6000)])
def test_tiles_equal_node_tiles(gpu_lib, grid, n, where):
    sc = _scene(grid, n, where)
    W = np.random.default_rng(n).standard_normal((8, n, 4)).astype(np.float32)
    W[1, :, 3] = 0.0
    out = []
    for forces in ([], [NOISE0]):
        sc.forces = forces
        e = make_engine(sc)
        e.substep(sc.dt, 2)
        grid_arrays = e.getGrid()
        e.adjointBegin(2, 2)
        e.forwardRecorded(sc.dt)
        e.setAdjoint(W)
        e.backward()
        out.append([e.getState(), e.getAdjoint(), *grid_arrays])
        e.adjointEnd()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_one_block_a_tile_equals_two(gpu_lib):
    rng = np.random.default_rng(2)
    a = _scene(61, 6000, "anywhere")
    fill = [falling_box(f"f{i}", 48, 3000, 2e4, 0.3, MaterialModel.ELASTIC, rng, corrected_svd=True) for i in range(48)]
    for s in fill:
        s.forces = []
    W = rng.standard_normal((8, a.n, 4)).astype(np.float32)
    W[1, :, 3] = 0.0
    got = []
    for e, total in ((make_engine(a), a.n), (make_batch_engine([a] + fill), a.n + sum(s.n for s in fill))):
        e.adjointBegin(3, 3)
        e.forwardRecorded(a.dt)
        full = np.zeros((8, total, 4), np.float32)
        full[:, :a.n] = W
        e.setAdjoint(full)
        e.backward()
        state = e.getState()[:, :a.n].copy()
        state[1, :, 3] = 0.0  # the batch's material ids are offset
        got.append((e.activeTileCount(), state, e.getAdjoint()[:, :a.n].copy()))
        e.adjointEnd()
    assert np.array_equal(got[0][1].view(np.uint32), got[1][1].view(np.uint32))
    assert np.array_equal(got[0][2].view(np.uint32), got[1][2].view(np.uint32))


def test_noise_four_threads_a_node_equal_one(gpu_lib):
    """A scene of at most 27 tiles alone and in a batch of more than 51; forces
    whose lattice points take several tables, one beyond any table."""
    rng = np.random.default_rng(4)
    a = _scene(24, 500, "anywhere")
    fill = [falling_box(f"f{i}", 48, 3000, 2e4, 0.3, MaterialModel.ELASTIC, rng, corrected_svd=True) for i in range(12)]
    a.forces = [mpm.GravityForce((0.0, 1.0, 0.0), -9.8), mpm.TurbulenceForce(strength=2.0, frequency=3.0, octaves=5, seed=1.0),
                mpm.TurbulenceForce(strength=1.0, frequency=7.0, octaves=4, seed=0.3),
                mpm.NoiseForce((0.0, 1.0, 0.0), 0.5, 5.0, 6, 0.7, 0.1), mpm.NoiseForce((1.0, 0.0, 0.0), 0.5, 900.0, 2, 0.7, 0.1)]
    W = rng.standard_normal((8, a.n, 4)).astype(np.float32)
    W[1, :, 3] = 0.0
    got = []
    for e, total in ((make_engine(a), a.n), (make_batch_engine([a] + fill), a.n + sum(s.n for s in fill))):
        e.substep(a.dt, 2)
        tiles = e.activeTileCount()
        e.adjointBegin(2, 2)
        e.forwardRecorded(a.dt)
        full = np.zeros((8, total, 4), np.float32)
        full[:, :a.n] = W
        e.setAdjoint(full)
        e.backward()
        state = e.getState()[:, :a.n].copy()
        state[1, :, 3] = 0.0  # the batch's material ids are offset
        got.append((tiles, state, e.getAdjoint()[:, :a.n].copy()))
        e.adjointEnd()
    assert got[0][0] <= 27 and got[1][0] > 51
    assert np.array_equal(got[0][1].view(np.uint32), got[1][1].view(np.uint32))
    assert np.array_equal(got[0][2].view(np.uint32), got[1][2].view(np.uint32))
