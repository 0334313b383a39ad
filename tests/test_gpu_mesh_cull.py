"""The mesh SDF's bounded search at its edges, bit for bit against the oracle's
pass over all triangles: grids smaller than a brick of 8^3 cells and not a
multiple of it, degenerate, sliver and non-finite triangles (never dropped,
and no bound may come from them), more candidates than a block's list holds,
long triangles whose missing edge region reaches across the grid, closed
surfaces far from most bricks."""
import numpy as np
import pytest

import oracle
from nebula_amd import mpm

pytestmark = pytest.mark.gpu


def _tris(v):
    v = np.asarray(v, np.float32).reshape(-1, 3, 3)
    n = np.cross(v[:, 1].astype(np.float64) - v[:, 0], v[:, 2].astype(np.float64) - v[:, 0])
    ln = np.linalg.norm(n, axis=1, keepdims=True)
    n = np.where(ln > 0, n / np.where(ln > 0, ln, 1), 0)
    return np.concatenate([n.astype(np.float32), v.reshape(-1, 9)], axis=1)


def _sphere(k, centre, radius):
    u, v = np.meshgrid(np.linspace(0, 2 * np.pi, 2 * k + 1), np.linspace(0, np.pi, k + 1), indexing="ij")
    p = np.stack([np.cos(u) * np.sin(v), np.cos(v), np.sin(u) * np.sin(v)], -1) * radius + centre
    a, b, c, d = p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]
    return np.concatenate([np.stack([a, b, c], 2).reshape(-1, 3, 3), np.stack([a, c, d], 2).reshape(-1, 3, 3)])


def _mesh(name):
    r = np.random.default_rng(len(name))
    if name == "few":
        return _tris(r.uniform(0.1, 0.9, (3, 3, 3)))
    if name == "sphere with degenerate poles":
        return _tris(_sphere(14, np.array([0.52, 0.47, 0.5]), 0.21))
    if name == "crowded ball":
        c = 0.5 + r.normal(0, 0.004, (6000, 1, 3))
        return _tris(c + r.normal(0, 0.002, (6000, 3, 3)))
    if name == "needles":
        a = r.uniform(0, 1, (500, 1, 3))
        return _tris(np.concatenate([a, a + r.uniform(-0.6, 0.6, (500, 1, 3)), a + r.uniform(-2e-3, 2e-3, (500, 1, 3))], 1))
    if name == "not finite":
        t = _tris(r.uniform(0.2, 0.8, (60, 3, 3)))
        t[7, 4], t[20, 9], t[33, 3:] = np.nan, np.inf, t[33, 3]
        return t
    t = _tris(r.uniform(0.3, 0.6, (900, 1, 3)) + r.uniform(-0.03, 0.03, (900, 3, 3)))
    return t


@pytest.mark.parametrize("exact", [False, True], ids=["reference", "exact"])
@pytest.mark.parametrize("res", [(4, 3, 4), (24, 24, 24), (17, 30, 9)], ids=str)
@pytest.mark.parametrize("name", ["few", "sphere with degenerate poles", "crowded ball", "needles", "not finite",
                                  "small in a large grid"])
def test_bounded_search_equals_the_pass_over_all(gpu_lib, name, res, exact):
    h = np.float32(1.0 / max(res))
    e = mpm.MPMEngine(mpm.MPMConfig(nx=0, ny=0, nz=0, domainSize=tuple(float(h) * n * 0.999 for n in res),
                                    cellSize=float(h), maxParticles=64))
    assert e.gridRes() == res
    tris = _mesh(name)
    e.setColliderMesh(tris, exact=exact)
    got = e.getColliderSDF()
    want = oracle.mesh_sdf(tris, res, float(h), exact=exact)
    diff = np.nonzero(got.view(np.uint32) != want.view(np.uint32))[0]
    assert diff.size == 0, f"{diff.size} of {got.size} cells differ: {got[diff[:4]]} vs {want[diff[:4]]}"
