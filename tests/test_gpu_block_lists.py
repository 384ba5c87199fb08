"""Listed substeps (k_bin_update) against a full binning of every substep: the
same state bit for bit, in scenes that reach the lists' edges."""

import numpy as np
import pytest

from tessera_amd.mpm import HipMpmResidentSession, HipMpmTransfers, MaterialModel, MpmParams, MpmWorld
from tessera_amd.scenes import _particles

pytestmark = pytest.mark.gpu

H, DT = 1.0 / 64, 1.0e-4


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


def blob(rng, n, first_cell, cells, velocity):
    lo = (np.array(first_cell, dtype=np.float64) + 0.55) * H
    pos = lo + rng.uniform(0.0, (cells - 0.1) * H, size=(n, 3))
    return pos, np.tile(np.asarray(velocity, dtype=np.float64) * H / DT, (n, 1))


# velocities in cells per substep
SCENES = {
    # 1,500 particles of one block cross a face within a few substeps into blocks that do not
    # exist: strays, and more than a block's 64 entries at once
    "dense_blob_into_new_blocks": [(1500, (16, 16, 16), 4, (0.3, 0.0, 0.0))],
    # corners and mixed signs: blocks that are neither a step up nor a step down
    "diagonal": [(300, (16, 16, 16), 4, (0.2, -0.2, 0.1)), (300, (32, 16, 16), 4, (-0.15, -0.2, -0.2))],
    # two bodies meet: particles come into blocks that hold others
    "meeting": [(700, (16, 16, 16), 8, (0.25, 0.0, 0.0)), (700, (26, 16, 16), 8, (-0.25, 0.0, 0.05))],
    # negative cells, and a lone particle per block
    "sparse": [(1, (-9 + 4 * k, -3, 5 * k), 1, (0.3, -0.1, 0.2)) for k in range(6)],
    # nothing leaves its block
    "at_rest": [(65, (16, 16, 16), 4, (0.0, 0.0, 0.0))],
}


@pytest.mark.parametrize("mode", ["fp32", "fixed64"])
@pytest.mark.parametrize("scene", sorted(SCENES))
def test_listed_substeps_equal_full_binning(transfers, scene, mode, monkeypatch):
    rng = np.random.default_rng(5)
    parts = [blob(rng, *b) for b in SCENES[scene]]
    pos, vel = np.concatenate([p for p, _ in parts]), np.concatenate([v for _, v in parts])
    pa = _particles(pos, vel, H / 4, 1.0e3, MaterialModel.fluid(1.0e2, 7.0, 0.0))
    pa.fixed[:: 97] = len(pos) > 97  # fixed particles stay on their block's list
    pa.transfer_color[1::2] = 1      # two colours: two blocks over the same cells
    world = MpmWorld(pa, MpmParams(cell_width=H, gravity=np.zeros(3), max_substep=DT, bounds=None))
    runs = {}
    for interval in (1, 16, 5):
        monkeypatch.setenv("TMPM_REORDER_INTERVAL", str(interval))
        s = HipMpmResidentSession(transfers, world, DT, mode)
        for k in (1, 19, 7, 13):  # submissions that end within and at the ends of the lists' spans
            s.step(k)
        assert s.valid and s.world().substeps == 40
        runs[interval] = (s.read_particles(), s.topology_stats())
        s.close()
    full, stats = runs[1]
    for interval in (16, 5):
        got, st = runs[interval]
        for f in ("position", "velocity", "affine", "deformation"):
            assert np.array_equal(getattr(got, f), getattr(full, f)), (interval, f)
        assert st == stats
