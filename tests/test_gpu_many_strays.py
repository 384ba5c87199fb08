"""Where substeps send many particles into blocks that do not exist, or more into
a block than its list has entries for, lists cost more than a full binning: the
session leaves them, and computes the same."""

import numpy as np
import pytest

from tessera_amd.mpm import HipMpmResidentSession, HipMpmTransfers, MaterialModel, MpmParams, MpmWorld
from tessera_amd.scenes import _particles

pytestmark = pytest.mark.gpu

H, DT = 1.0 / 64, 1.0e-4


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


def cloud(n, cells, speed, spread):
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, cells, size=(n, 3))
    vel = (np.array([0.8, -0.5, 0.33]) + spread * (pos / cells - 0.5)) * speed
    pa = _particles(pos * H, vel * H / DT, H / 4, 1.0e3, MaterialModel.elastic(1.0e-9, 0.3))
    return MpmWorld(pa, MpmParams(cell_width=H, gravity=np.zeros(3), max_substep=DT, bounds=None))


# 30,000 particles, about one a block: some 1,100 strays a substep.  60,000, 16 a cell: about 125 of
# a block's 1,024 leave it for the next one, which has 64 entries.  The other scenes have next to none.
@pytest.mark.parametrize("n,cells,speed,spread,leaves", [(30000, 128, 0.3, 0.3, True), (60000, 15.5, 0.3, 0.0, True),
                                                         (30000, 128, 0.0, 0.3, False), (30000, 24, 0.1, 0.3, False)])
def test_lists_are_left_where_many_particles_stray(transfers, n, cells, speed, spread, leaves, monkeypatch):
    runs = []
    for interval in (1, 16):
        monkeypatch.setenv("TMPM_REORDER_INTERVAL", str(interval))
        s = HipMpmResidentSession(transfers, cloud(n, cells, speed, spread), DT)
        s.set_timing(True)
        for _ in range(12):
            s.step(16)
        runs.append(s.read_particles())
        calls = {k: v[1] for k, v in s.kernel_times().items()}
        s.close()
    for f in ("position", "velocity", "affine", "deformation"):
        assert np.array_equal(getattr(runs[0], f), getattr(runs[1], f)), f
    listed, full = calls.get("k_bin_update", 0), calls["k_bin_insert"]
    assert listed + full == 192
    # in the first of the 12 intervals, then two substeps each of the 3rd, 6th and 11th
    assert (listed <= 15 + 3 * 2) if leaves else (listed == 12 * 15)
