"""The readback of a plain session (k_gather_state, copied and widened in
pieces of 144,631 records) against the particle snapshot of the same state."""

import numpy as np
import pytest

from tessera_amd.mpm import HipMpmResidentSession, HipMpmTransfers, MaterialModel, MpmParams, MpmWorld
from tessera_amd.scenes import _particles
from tests.hip_util import DeviceBuffer

pytestmark = pytest.mark.gpu

PIECE = ((16 << 20) // 4 - 16) // 29


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


@pytest.mark.parametrize("n", [1, 257, PIECE - 1, PIECE, PIECE + 1, 2 * PIECE + 3])
def test_readback_equals_the_snapshot(transfers, n):
    rng = np.random.default_rng(n)
    h = 1.0 / 64
    pos = np.float32(rng.uniform(0.2, 0.8, size=(n, 3))).astype(np.float64)
    vel = np.float32(rng.normal(0.0, 0.3, size=(n, 3))).astype(np.float64)
    pa = _particles(pos, vel, h / 8, 1.0e3, MaterialModel.elastic(1.0e4, 0.3))
    pa.enabled[3::7] = False
    pa.fixed[5::11] = True
    s = HipMpmResidentSession(transfers, MpmWorld(pa, MpmParams(cell_width=h, max_substep=1e-4)), 1e-4)
    for steps in (1, 2):
        s.step(steps)
        got = s.read_particles()
        buf = DeviceBuffer(32 * n)
        assert s.encode_particle_snapshot(buf.ptr, buf.nbytes) == n
        rec = buf.read(np.float32).reshape(n, 8)
        on = pa.enabled
        assert np.array_equal(got.position[on & ~pa.fixed], rec[on & ~pa.fixed, :3])
        assert np.array_equal(got.velocity[on], rec[on, 4:7])
        assert np.array_equal(got.position[~on | pa.fixed], pos[~on | pa.fixed])
        assert np.array_equal(got.velocity[~on], vel[~on]) and not got.velocity[on & pa.fixed].any()
        assert not np.array_equal(got.deformation[0], np.eye(3)) or n == 1
        assert np.all(got.affine[pa.fixed & on] == 0.0) and np.array_equal(got.mass, pa.mass)
        assert np.array_equal(got.enabled, pa.enabled) and np.array_equal(got.fixed, pa.fixed)
    s.close()
