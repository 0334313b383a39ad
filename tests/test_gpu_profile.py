"""nb_mpm_profile_substeps books the FP64 fallback's work under its own name, for
cubes on both sides of the one-launch tile pass and for batches, and leaves the
results of unprofiled substeps."""
import numpy as np
import pytest

from nebula_amd.mpm import MaterialModel
from nebula_amd.scenes import falling_box, make_batch_engine, make_engine
from test_gpu_batch import _scenes

pytestmark = pytest.mark.gpu


def _flat(sc):
    """Equal singular values: every Drucker-Prager particle takes the fallback."""
    sc.fields[2:5, :, :3] = (np.eye(3) * (0.98, 0.95, 0.98))[:, None]
    return sc


def _make(kind):
    if kind == "batch":
        scenes = [_flat(s) for s in _scenes()]
        return (lambda: make_batch_engine(scenes)), scenes[0].dt
    sc = _flat(falling_box("p", 64 if kind == "small" else 256, 30000, 3e4, 0.3, MaterialModel.DRUCKER_PRAGER,
                           np.random.default_rng(1)))
    return (lambda: make_engine(sc)), sc.dt


@pytest.mark.parametrize("kind", ["small", "large", "batch"])
def test_fallback_is_booked_by_name(gpu_lib, kind):
    make, dt = _make(kind)
    plain, timed, off = make(), make(), make()
    plain.substep(dt, 5)
    prof = timed.profileSubsteps(dt, 5)
    calls = timed.profileCalls()
    assert calls["g2p_fb"] == 6 and calls["g2p"] == 5, calls
    assert np.array_equal(plain.getState().view(np.uint32), timed.getState().view(np.uint32))
    off.setSvdFallback(False)
    without = off.profileSubsteps(dt, 5)
    print({k: (round(v, 3), round(without.get(k, 0.0), 3)) for k, v in prof.items()}, flush=True)
    assert off.profileCalls().get("g2p_fb", 0) == 0
    # six launches that find work are not less than two times what a launch costs
    assert prof["g2p_fb"] > 0.03
