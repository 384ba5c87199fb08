"""A batch scene that fails within a submission stops with the next substep,
listed or fully binned: what the device holds of it does not move any more."""

import numpy as np
import pytest

from tessera_amd.mpm import HipMpmBatch, HipMpmResidentSession, HipMpmTransfers
from tests.hip_util import DeviceBuffer
from tests.test_gpu_batch import dts_for, mixed_worlds

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


def snapshot(b, n):
    buf = DeviceBuffer(32 * n)
    HipMpmResidentSession.encode_particle_snapshot(b, buf.ptr, buf.nbytes)
    return buf.read(np.float32).reshape(n, 8)


@pytest.mark.parametrize("mode", ["fp32", "fixed64"])
@pytest.mark.parametrize("tail", [1, 9])
def test_a_failed_scene_stops_in_listed_substeps(transfers, mode, tail, monkeypatch):
    worlds = mixed_worlds()[:3]
    dts = dts_for(worlds)
    n = sum(len(w.particles) for w in worlds)
    shots = {}
    # From the 34th substep on: no lists any more without a reorder at hand (fully binned), and
    # listed up to the reorder before the 49th (a reorder drops what is not binned).
    for interval in (1000000, 16):
        monkeypatch.setenv("TMPM_REORDER_INTERVAL", str(interval))
        b = HipMpmBatch(transfers, worlds, dts, mode)
        b.step(34)
        m = float(worlds[1].particles.mass[0])
        b.set_particle_force(1, 0, [200.0 * m / dts[1], 0.0, 0.0])  # past the CFL bound in the next substep
        b.submit_steps(1 + tail)
        shots[interval] = snapshot(b, n)
        b.synchronize()
        assert [b.scene_error(k) is None for k in range(3)] == [True, False, True]
        b.close()
    assert np.array_equal(shots[1000000], shots[16])
