"""The status of a readback is that of the session's own state: what an earlier
session left in device memory does not enter it."""

import numpy as np
import pytest

from tessera_amd.mpm import GpuMpmError, HipMpmResidentSession, HipMpmTransfers, MaterialModel, MpmParams, MpmWorld
from tessera_amd.scenes import _particles

pytestmark = pytest.mark.gpu

H, DT = 1.0 / 64, 1.0e-4


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


def world(n):
    rng = np.random.default_rng(n)
    pa = _particles(rng.uniform(0.3, 0.6, size=(n, 3)), np.zeros((n, 3)), H / 4, 1.0e3,
                    MaterialModel.elastic(1.0e3, 0.3))
    return MpmWorld(pa, MpmParams(cell_width=H, gravity=np.zeros(3), max_substep=DT, bounds=None))


# from a few kilobytes to a readback in two pieces
@pytest.mark.parametrize("n", [2, 3000, 150000])
@pytest.mark.parametrize("readbacks", [1, 3])
def test_a_session_after_a_non_finite_one_is_healthy(transfers, n, readbacks):
    bad = HipMpmResidentSession(transfers, world(n), DT)
    for _ in range(readbacks - 1):
        bad.step(1)
    bad.set_particle_force(0, [3.0e38, 0.0, 0.0])  # the velocity overflows: no finite position
    with pytest.raises(GpuMpmError):
        bad.step(1)
    assert not bad.valid
    bad.close()
    for _ in range(2):  # the sizes are the failed session's: its memory may come back as it was left
        good = HipMpmResidentSession(transfers, world(n), DT)
        for _ in range(readbacks + 2):
            good.step(1)
        assert good.valid and np.isfinite(good.read_particles().position).all()
        good.close()


@pytest.mark.parametrize("readbacks", [1, 2])
def test_a_non_finite_state_is_reported_at_its_own_readback(transfers, readbacks):
    s = HipMpmResidentSession(transfers, world(500), DT)
    for _ in range(readbacks - 1):
        s.step(1)
    last = s.read_particles()
    s.set_particle_force(7, [0.0, -3.0e38, 0.0])
    with pytest.raises(GpuMpmError):
        s.step(1)
    # the last synchronized world stays readable
    got = s.read_particles()
    for f in ("position", "velocity", "affine", "deformation"):
        assert np.array_equal(getattr(got, f), getattr(last, f)), f
    s.close()
