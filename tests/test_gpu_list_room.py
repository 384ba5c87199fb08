"""Scenes that visit more blocks between two full binnings than there is memory
for beside the emptied ones, though every substep's own blocks fit: they run on,
and their state is that of a full binning of every substep, bit for bit."""

import numpy as np
import pytest

from tessera_amd.mpm import HipMpmResidentSession, HipMpmTransfers, MaterialModel, MpmParams, MpmWorld
from tessera_amd.scenes import _particles

pytestmark = pytest.mark.gpu

H, DT = 1.0 / 64, 1.0e-4


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


def drifting(rng):
    # 1,000 lone particles, 12 cells apart, on a diagonal near the CFL bound: 3,708 blocks visited
    # in 16 substeps, room for 2,000
    g = np.stack(np.meshgrid(*[np.arange(10)] * 3, indexing="ij"), -1).reshape(-1, 3) * 12.0 + 17.6
    return g + rng.uniform(0.0, 2.0, size=g.shape), np.tile([0.22, -0.22, 0.22], (1000, 1))


def burst(rng):
    # 300 clumps fly out of one block: within the 4,096 grid blocks that are allowed at each of 256
    # substeps, but not within the room for 6,144 by the blocks visited in 32
    c = 16.6 + rng.uniform(0.0, 3.8, size=(300, 3))
    v = c - 18.5
    v *= 0.39 / np.linalg.norm(v, axis=1).max()
    pos = np.repeat(c, 6, axis=0)
    return pos + rng.uniform(0.0, 0.01, size=pos.shape), np.repeat(v, 6, axis=0)


@pytest.mark.parametrize("mode", ["fp32", "fixed64"])
@pytest.mark.parametrize("scene,interval,submissions", [(drifting, 16, (40,)), (burst, 32, (64,) * 4)])
def test_visited_blocks_beyond_the_room(transfers, scene, interval, submissions, mode, monkeypatch):
    cells, v = scene(np.random.default_rng(3))
    pa = _particles(cells * H, v * H / DT, H / 4, 1.0e3, MaterialModel.elastic(1.0e-9, 0.3))
    world = MpmWorld(pa, MpmParams(cell_width=H, gravity=np.zeros(3), max_substep=DT, bounds=None))
    runs = []
    for every in (1, interval):
        monkeypatch.setenv("TMPM_REORDER_INTERVAL", str(every))
        s = HipMpmResidentSession(transfers, world, DT, mode)
        for k in submissions:  # nothing grows the tables in between
            s.submit_steps(k)
        s.synchronize()
        runs.append((s.read_particles(), s.topology_stats()))
        s.close()
    (full, stats), (got, st) = runs
    assert st == stats
    for f in ("position", "velocity", "affine", "deformation"):
        assert np.array_equal(getattr(got, f), getattr(full, f)), f
