"""Device memory of an engine: what the header says, and none for the work items of
small scenes in a batch that never takes them.  Each engine is measured in a process
of its own, where the runtime holds nothing that an earlier engine gave back."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import ctypes as C, sys
sys.path.insert(0, sys.argv[1])
from nebula_amd import hip, mpm
def free():
    f, t = C.c_size_t(), C.c_size_t()
    hip.synchronize()
    hip.check(hip.runtime().hipMemGetInfo(C.byref(f), C.byref(t)), "hipMemGetInfo")
    return f.value
scenes, n = int(sys.argv[2]), int(sys.argv[3])
first = mpm.MPMEngine(mpm.MPMConfig(nx=0, ny=0, nz=0, domainSize=(0.5,) * 3, cellSize=1.0 / 64, maxParticles=64))
a = free()
if scenes:
    e = mpm.MPMEngine.batch([mpm.BatchScene((0.5,) * 3, 1.0 / 64, n // scenes) for _ in range(scenes)])
else:
    e = mpm.MPMEngine(mpm.MPMConfig(nx=0, ny=0, nz=0, domainSize=(1.0,) * 3, cellSize=1.0 / 64, maxParticles=n))
print(a - free())
"""


@pytest.mark.parametrize("scenes, particles, items", [(16, 262144, 262144), (17, 17 * 15000, 0), (12, 12 * 21846, 0),
                                                      (0, 200000, 200000), (0, 600000, 262144)])
def test_device_memory(gpu_lib, scenes, particles, items):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CHILD, root, str(scenes), str(particles)], capture_output=True, text=True,
                       timeout=100, check=True)
    used = int(r.stdout.split()[-1])
    cubes, edge = (scenes, 32) if scenes else (1, 64)
    tiles = cubes * (edge // 8) ** 3
    said = 356 * particles + 448 * items + 42 * cubes * edge ** 3 + 16000 * min(tiles, particles)
    print(f"  {scenes} scenes, {particles} particles: {used / 2**20:.1f} MiB, said {said / 2**20:.1f}", flush=True)
    assert abs(used - said) < 32 << 20  # nine allocations in pages of 2 MiB and more
