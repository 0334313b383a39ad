"""The mesh SDF's bounded search where rounding moves a triangle's closest point
by more than a fixed share of the distance: strips up to 10,000 cells long and up
to 80 times longer than wide, and triangles far smaller than a cell seen from
across the grid; and meshes too small or too flat for the search.  Bit for bit
against the oracle's pass over all triangles."""
import time

import numpy as np
import pytest

import oracle
from nebula_amd import mpm
from test_gpu_mesh_cull import _tris

pytestmark = pytest.mark.gpu


def _strips(length, ratio, res, count, r):
    """Triangles of the given length in cells and length / height, side by side on
    a tilted plane through the grid's middle, a little off it."""
    d = r.normal(size=3)
    d /= np.linalg.norm(d)
    n = np.cross(d, r.normal(size=3))
    n /= np.linalg.norm(n)
    w = np.cross(n, d)
    L, W = length / res, length / res / ratio
    out = []
    for i in range(count):
        c = 0.5 + w * (i - count / 2) * min(W, 1.5 / count) + d * r.uniform(-0.4, 0.4) * L + n * r.normal() * 0.02
        out.append([c - d * L / 2, c + d * L / 2, c + w * W + d * r.uniform(-0.5, 0.5) * L])
    return _tris(out)


def _specks(ratio, res, count, r):
    """Triangles of 0.002 to 0.5 cells on a small ball near a corner."""
    s = (0.002 * 250.0 ** r.random((count, 1, 1))) / res
    n = r.normal(size=(count, 3))
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    d = np.cross(n, r.normal(size=(count, 3)))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    w = np.cross(n, d)
    v = np.stack([0 * d, d, r.random((count, 1)) * d + w / ratio], 1) * s
    return _tris(v + (0.2 + 0.06 * n)[:, None])


def _check(tris, res, exact):
    h = np.float32(1.0 / res)
    e = mpm.MPMEngine(mpm.MPMConfig(nx=0, ny=0, nz=0, domainSize=(0.999,) * 3, cellSize=float(h), maxParticles=64))
    assert e.gridRes() == (res,) * 3
    e.setColliderMesh(tris, exact=exact)
    got = e.getColliderSDF()
    want = oracle.mesh_sdf(tris, (res,) * 3, float(h), exact=exact)
    diff = np.nonzero(got.view(np.uint32) != want.view(np.uint32))[0]
    assert diff.size == 0, f"{diff.size} of {got.size} cells differ: {got[diff[:4]]} vs {want[diff[:4]]}"


@pytest.mark.parametrize("exact", [False, True], ids=["reference", "exact"])
@pytest.mark.parametrize("ratio", [10, 30, 80])
@pytest.mark.parametrize("length", [100, 1000, 10000])
def test_long_strips(gpu_lib, length, ratio, exact):
    for res in (32, 64):
        _check(_strips(length, ratio, res, 60, np.random.default_rng(length + ratio)), res, exact)


@pytest.mark.parametrize("exact", [False, True], ids=["reference", "exact"])
@pytest.mark.parametrize("ratio", [2, 20, 90])
def test_small_triangles_from_afar(gpu_lib, ratio, exact):
    _check(_specks(ratio, 64, 150, np.random.default_rng(ratio)), 64, exact)


@pytest.mark.parametrize("exact", [False, True], ids=["reference", "exact"])
@pytest.mark.parametrize("n, flat", [(15, 0), (16, 16), (17, 0), (17, 8), (18, 9), (18, 10), (400, 199), (400, 200),
                                     (400, 201), (1500, 1500)])
def test_few_and_mostly_unbounded_meshes(gpu_lib, n, flat, exact):
    """Around the sizes and the share of triangles without height where every cell
    measures all of them."""
    r = np.random.default_rng(n + flat)
    v = r.uniform(0.1, 0.9, (n, 1, 3)) + r.uniform(-0.1, 0.1, (n, 3, 3))
    v[:flat, 2] = 0.5 * (v[:flat, 0] + v[:flat, 1])
    _check(_tris(v[r.permutation(n)]), 32, exact)


def test_unbounded_triangles_cost_no_more_than_measuring_them(gpu_lib):
    """2000 triangles of no height on 128^3 cells: 3.2 ms when every cell just measures
    all, 7.7 when each is first looked up in the search's lists."""
    p = np.random.default_rng(0).uniform(0, 1, (2000, 1, 3))
    e = mpm.MPMEngine(mpm.MPMConfig(nx=0, ny=0, nz=0, domainSize=(1.0,) * 3, cellSize=1.0 / 128, maxParticles=64))
    tris, best = _tris(np.repeat(p, 3, 1)), 1e9
    for _ in range(8):
        t = time.perf_counter()
        e.setColliderMesh(tris)
        best = min(best, time.perf_counter() - t)
    print(f"  {best * 1e3:.2f} ms", flush=True)
    assert best < 5.2e-3
