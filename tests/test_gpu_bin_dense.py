"""The bin of tiles that hold more particles than its LDS stage (6144): cell ranges
that end at, before and after the stage, cells that fill it alone and cells beyond
it, bit for bit against a stable numpy sort; and in the time of a few passes over
the tile, where ordering cell by cell took twice the time of tiles that fit."""
import time

import numpy as np
import pytest

from test_gpu_bin_paths import _check_bins, _engine

pytestmark = pytest.mark.gpu


def _cells(counts, rng):
    """Positions with counts[c] particles in the c-th cell of a tile (x fastest) of a
    32^3 grid, in no order."""
    counts = np.asarray(counts)
    c = np.arange(len(counts))
    ijk = np.stack([c % 8, c // 8 % 8, c // 64], 1) + 8
    p = (np.repeat(ijk, counts, axis=0) + rng.uniform(0.1, 0.9, (counts.sum(), 3))) / 32
    return p[rng.permutation(len(p))].astype(np.float32)


@pytest.mark.parametrize("name", ["13 each", "40 each", "ends at the stage", "one over", "gaps", "alone", "beyond", "all"])
def test_dense_tiles(gpu_lib, name):
    rng = np.random.default_rng(len(name))
    c = {"13 each": np.full(512, 13), "40 each": np.full(512, 40),
         "ends at the stage": np.repeat([64, 0, 96], [96, 100, 70]),  # 6144 and more
         "one over": np.r_[np.full(95, 64), 65, np.full(95, 64), 63, 65, np.zeros(300, int), 9],
         "gaps": np.where(rng.random(512) < 0.1, 300, 0),
         "alone": np.r_[0, 6144, 0, 6144, 3, 6144],
         "beyond": np.r_[5, 6145, 0, 1, 20011, 7, 6143, 8193, 2],
         "all": np.r_[np.zeros(511, int), 30000]}[name]
    pos = _cells(c, rng)
    e, h = _engine(pos, (32, 32, 32))
    e.runBin()
    _check_bins(e, pos, h, (32, 32, 32))


def _bin_time(per_cell):
    rng = np.random.default_rng(per_cell)
    edge = round((1048576 / per_cell) ** (1 / 3))
    ijk = np.stack(np.unravel_index(np.arange(edge ** 3), (edge,) * 3), 1) + 4
    pos = (np.repeat(ijk, per_cell, axis=0) + rng.uniform(0.1, 0.9, (per_cell * edge ** 3, 3))) / 64
    e, _ = _engine(pos.astype(np.float32), (64, 64, 64))
    best = 1e9
    for _ in range(30):
        t = time.perf_counter()
        e.runBin()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("per_cell", [16, 32])
def test_dense_tiles_do_not_serialise(gpu_lib, per_cell):
    """A million particles: 69 us at 8 a cell; at 16 and 32, 67 and 75 with a cell a
    thread, 138 and 180 with a cell a wave after the other."""
    a, b = _bin_time(8), _bin_time(per_cell)
    print(f"  8 a cell {a * 1e6:.0f} us, {per_cell} a cell {b * 1e6:.0f} us", flush=True)
    assert b < 1.6 * a
