"""The bin's two-level sort where its paths change, bit for bit against a stable
numpy sort of the cell keys: tiles of any size against the LDS stage (6144),
cells up to a wave and beyond, more than 2^23 particles (two-word entries),
cubes on both sides of the one-launch tile pass, and counts left over from a
state that was replaced."""
import numpy as np
import pytest

from nebula_amd import mpm
from nebula_amd.mpm import MaterialModel
from nebula_amd.scenes import elastic_block_64, falling_box, make_batch_engine, make_engine

pytestmark = pytest.mark.gpu


def _engine(pos, res):
    n, h = len(pos), 1.0 / max(res)
    e = mpm.MPMEngine(mpm.MPMConfig(nx=0, ny=0, nz=0, domainSize=tuple(r * h for r in res), cellSize=h, maxParticles=n))
    f = np.zeros((8, n, 4), np.float32)
    f[0, :, :3], f[0, :, 3] = pos, h ** 3 / 8
    f[2, :, 0] = f[3, :, 1] = f[4, :, 2] = 1.0
    e.setState(f)
    return e, h


def _check_bins(e, pos, h, res):
    keys, srt, cnt, end = e.getBins()
    ijk = np.clip((pos / np.float32(h)).astype(np.int64), 0, np.array(res) - 1)
    want = mpm.mortonEncodeArray(ijk[:, 0], ijk[:, 1], ijk[:, 2]).astype(np.uint32)
    assert np.array_equal(keys, want)
    assert np.array_equal(srt, np.argsort(want, kind="stable").astype(np.uint32))
    full = np.bincount(want, minlength=cnt.size).astype(np.uint32)
    assert np.array_equal(cnt, full) and np.array_equal(end, np.cumsum(full).astype(np.uint32))


@pytest.mark.parametrize("per_tile", [1, 63, 512, 2047, 2049, 6143, 6144, 6145, 9000])
@pytest.mark.parametrize("spread", ["cells", "few"])
def test_tiles_around_the_stage(gpu_lib, per_tile, spread):
    res = (40, 24, 33)
    rng = np.random.default_rng(per_tile)
    h = 1.0 / 40
    tiles = [(0, 0, 0), (4, 2, 3), (1, 0, 2)]
    pos = []
    for t in tiles:
        cells = rng.integers(0, 8, (per_tile, 3))
        if spread == "few":  # cells of 2, 60 to 70 and many particles
            pick = np.array([[1, 1, 1], [2, 3, 4], [7, 0, 5], [6, 6, 0]])
            cells = pick[np.minimum(np.arange(per_tile) // 65, 3)]
        pos.append((np.array(t) * 8 + cells + rng.uniform(0.1, 0.9, (per_tile, 3))) * h)
    pos = np.concatenate(pos)
    pos = np.minimum(pos, (np.array(res) - 0.5) * h)
    pos = pos[rng.permutation(len(pos))].astype(np.float32)
    e, h = _engine(pos, res)
    e.runBin()
    _check_bins(e, pos, h, res)


@pytest.mark.parametrize("res", [(8, 8, 8), (5, 7, 3), (64, 64, 64), (128, 100, 77), (129, 40, 30), (256, 16, 200)], ids=str)
def test_cubes_around_the_one_launch_tile_pass(gpu_lib, res):
    rng = np.random.default_rng(sum(res))
    pos = (rng.random((30011, 3)) * np.array(res) / max(res)).astype(np.float32)
    pos[:9000] = pos[:9000] * 0.1
    e, h = _engine(pos, res)
    e.runBin()
    _check_bins(e, pos, h, res)


def test_more_particles_than_packed_entries_hold(gpu_lib):
    rng = np.random.default_rng(8)
    n, res = (1 << 23) + 70001, (128, 128, 128)
    pos = rng.random((n, 3), np.float32)
    e, h = _engine(pos, res)
    e.runBin()
    _check_bins(e, pos, h, res)


def test_counts_of_a_replaced_state_are_dropped(gpu_lib):
    sc = elastic_block_64(res=32)
    a, b = make_engine(sc), make_engine(sc)
    moved = sc.fields.copy()
    moved[0, :, 0] += np.float32(0.21)
    b.setState(moved)
    b.substep(sc.dt, 3)
    a.substep(sc.dt, 2)          # leaves counts for a next substep
    a.setState(moved)            # which never comes
    a.substep(sc.dt, 1)
    a.runBin()                   # and a bin between substeps
    _check_bins(a, a.getField(0)[:, :3], 1.0 / 32, (32, 32, 32))
    a.substep(sc.dt, 1)
    a.graphSubstep(sc.dt, 1)
    assert np.array_equal(a.getState().view(np.uint32), b.getState().view(np.uint32))
    a.runBin()
    a.runP2G(sc.dt)
    a.runGridUpdate(sc.dt)
    a.runG2P(sc.dt)              # keys, no counts
    a.substep(sc.dt, 2)
    b.substep(sc.dt, 3)
    assert np.array_equal(a.getField(0).view(np.uint32), b.getField(0).view(np.uint32))


def test_batch_beyond_the_summed_blocks(gpu_lib):
    """70 scenes of 128^3 cubes: 286,720 tiles, 1,120 blocks of them."""
    rng = np.random.default_rng(5)
    scenes = [falling_box(f"s{i}", 96, 300 + 7 * i, 2e4, 0.3, MaterialModel.ELASTIC if i % 2 else
                          MaterialModel.DRUCKER_PRAGER, rng) for i in range(70)]
    e = make_batch_engine(scenes)
    e.substep(scenes[0].dt, 4)
    got = e.getState()
    for i in (0, 1, 33, 68, 69):
        s = make_engine(scenes[i])
        s.substep(scenes[i].dt, 4)
        _, first, count = e.sceneInfo(i)
        one, part = s.getState(), got[:, first:first + count].copy()
        part[1, :, 3] = one[1, :, 3]  # the batch's material ids are offset
        assert np.array_equal(part.view(np.uint32), one.view(np.uint32)), i
