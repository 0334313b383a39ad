"""nb_hash_build and nb_hash_build_noalloc write nothing of ``sorted`` past the
used particles, whatever share of the slots is unused, at hashes below, at and
above the sizes where the build takes scratch memory."""
import numpy as np
import pytest

import oracle
from nebula_amd import hip
from nebula_amd.hash import build, make_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("n, used", [(1, 0), (3, 1), (64, 0), (64, 2), (100, 3), (5000, 70), (5000, 5000)])
@pytest.mark.parametrize("res", [4, 16, 32, 64, 128])
def test_tail_of_sorted_is_left_alone(gpu_lib, res, n, used, noalloc):
    rng = np.random.default_rng(res + n)
    p = np.zeros((n, 4), np.float32)
    p[:, :3] = rng.random((n, 3))
    tf = np.full(n, 6, np.uint32)
    tf[rng.permutation(n)[:used]] = 1
    grid = make_grid((0, 0, 0), 1.0 / res, (res,) * 3)
    tail = np.arange(n, dtype=np.uint32) + 0xABC00000
    d = [hip.DeviceArray.from_host(a) for a in (p, tf, np.zeros(res ** 3, np.uint32), np.zeros(res ** 3, np.uint32), tail)]
    build(grid, d[0].ptr, d[1].ptr, n, d[2].ptr, d[3].ptr, d[4].ptr, noalloc=noalloc)
    hip.synchronize()
    cnt, off, srt = (a.download() for a in d[2:])
    want = oracle.hash_build(p, tf, (0, 0, 0), 1.0 / res, (res,) * 3)
    assert np.array_equal(cnt, want[0]) and np.array_equal(off, want[1])
    assert np.array_equal(srt[:used], want[2])
    assert np.array_equal(srt[used:], tail[used:])
