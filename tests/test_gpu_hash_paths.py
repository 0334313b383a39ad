"""The hash build where its launch rules and per-wave paths change, bit for bit
against the oracle: cells around the sizes that go from a thread's sort to
its wave's to a block's (16, 64, 256), runs of equal cells of every length and
across waves, particles in no order, four cells a thread against one, hashes
beyond 4096 scan blocks, and with and without the crowded list, its overflow
included."""
import numpy as np
import pytest

from test_gpu_hash import _check

pytestmark = pytest.mark.gpu


def _points(cells, counts, res, rng):
    ijk = np.stack(np.unravel_index(cells, (res, res, res)), 1)
    x = np.repeat(ijk, counts, axis=0) + rng.uniform(0.05, 0.95, (int(counts.sum()), 3))
    p = np.zeros((len(x), 4), np.float32)
    p[:, :3] = x / res
    return p


@pytest.mark.parametrize("res", [8, 32, 64], ids=lambda r: f"{r}^3")
@pytest.mark.parametrize("order", ["cells", "mixed", "alternating"])
def test_cell_sizes_around_the_sort_paths(gpu_lib, res, order):
    rng = np.random.default_rng(res)
    sizes = np.array([1, 2, 4, 5, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 600])
    k = np.tile(sizes, 6)
    cells = rng.choice(res ** 3, k.size, replace=False)
    p = _points(cells, k, res, rng)
    if order == "mixed":
        p = p[rng.permutation(len(p))]
    elif order == "alternating":  # equal cells never neighbours in storage
        p = p[np.argsort(np.arange(len(p)) % 61, kind="stable")]
    tf = np.where(rng.random(len(p)) < 0.1, 6, 0).astype(np.uint32)
    _check(f"{order} {res}", p, tf, (0, 0, 0), 1.0 / res, (res, res, res))


def test_more_than_4096_scan_blocks(gpu_lib):
    rng = np.random.default_rng(3)
    p = np.zeros((100001, 4), np.float32)
    p[:, :3] = rng.uniform(0, 1, (len(p), 3)) * np.array([300, 10, 500]) / 500
    p[:5000, :3] = p[0, :3]
    _check("512^3 cells", p, None, (0, 0, 0), 1.0 / 500, (300, 10, 500))


@pytest.mark.parametrize("res, many", [(64, 3000), (128, 3000), (128, 66000)])
def test_cells_beyond_a_wave_with_and_without_their_list(gpu_lib, res, many):
    """64^3 cells: no list; 128^3: the list, and with 66,000 cells its overflow."""
    rng = np.random.default_rng(4)
    lo = 0 if many > 10000 else 5000  # a run of neighbouring crowded cells
    cells = rng.choice(res ** 3, many, replace=False) if many > 10000 else np.arange(lo, lo + many)
    ijk = np.stack(np.unravel_index(cells, (res, res, res)), 1)
    p = np.zeros((many * 257, 4), np.float32)
    p[:, :3] = (np.repeat(ijk, 257, axis=0) + rng.random((many * 257, 3), np.float32) * 0.9 + 0.05) / res
    p = p[rng.permutation(len(p))]
    cnt, _, _ = _check(f"{many} cells of 257", p, None, (0, 0, 0), 1.0 / res, (res, res, res))
    assert np.sum(cnt > 256) == many


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 5000])
@pytest.mark.parametrize("order", ["runs", "mixed"])
def test_places_kept_from_the_count(gpu_lib, n, order):
    """Beyond 2^18 cells the count keeps the particles' places: runs of equal cells
    within and across waves, unused slots between them, and no order at all."""
    rng = np.random.default_rng(n)
    cells = np.repeat(rng.choice(128 ** 3, n, replace=False), rng.integers(1, 90, n))[:n]
    p = _points(cells, np.ones(n, int), 128, rng)
    if order == "mixed":
        p = p[rng.permutation(n)]
    tf = np.where(rng.random(n) < 0.2, 6, 0).astype(np.uint32)
    _check(f"{order} {n}", p, tf, (0, 0, 0), 1.0 / 128, (128, 128, 128))
