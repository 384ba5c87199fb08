"""Launch widths and grids that follow the block count: every width computes the
same state bit for bit, on both sides of each line, and a scene whose blocks
multiply between synchronizations is stepped by the smaller grid."""

import numpy as np
import pytest

from tessera_amd.mpm import HipMpmResidentSession, HipMpmTransfers, MaterialModel, MpmParams, MpmWorld
from tessera_amd.scenes import _particles

pytestmark = pytest.mark.gpu

H, DT = 1.0 / 64, 1.0e-4


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


def world_of(pos, vel, material):
    pa = _particles(pos, vel, H / 4, 1.0e3, material)
    return MpmWorld(pa, MpmParams(cell_width=H, gravity=np.array([0.0, -9.8, 0.0]), max_substep=DT, bounds=None))


def blocks_scene(rng, blocks, per_block, dense):
    """`blocks` blocks of 4^3 cells, `per_block` particles each; the first holds `dense` more."""
    edge = int(np.ceil(blocks ** (1.0 / 3.0)))
    k = np.arange(blocks)
    corner = 4 * np.stack([k // (edge * edge), k // edge % edge, k % edge], axis=1)
    of = np.concatenate([np.repeat(k, per_block), np.zeros(dense, dtype=int)])
    cells = corner[of] + rng.uniform(0.6, 4.4, size=(len(of), 3))
    return cells * H, rng.normal(0.0, 0.02 * H / DT, size=(len(of), 3))


@pytest.mark.parametrize("material", ["elastic", "sand"])
@pytest.mark.parametrize("mode", ["fp32", "fixed64"])
@pytest.mark.parametrize("blocks,per_block,dense", [(1, 1, 0), (1, 513, 600), (257, 64, 0), (257, 65, 300), (512, 9, 700),
                                                    (513, 129, 0), (1024, 5, 300), (1025, 3, 0)])
def test_widths_compute_the_same_state(transfers, blocks, per_block, dense, mode, material, monkeypatch):
    rng = np.random.default_rng(blocks + per_block)
    pos, vel = blocks_scene(rng, blocks, per_block, dense)
    m = MaterialModel.elastic(1.0e4, 0.3) if material == "elastic" else MaterialModel.sand(1.0e4, 0.3, 0.6, 0.0)
    runs = []
    for width in (None, "64"):
        if width:
            monkeypatch.setenv("TMPM_P2G_THREADS", width)
            monkeypatch.setenv("TMPM_PBLOCK_THREADS", width)
        s = HipMpmResidentSession(transfers, world_of(pos, vel, m), DT, mode)
        for k in (1, 18):
            s.step(k)
        runs.append(s.read_particles())
        s.close()
    a, b = runs
    for name in ("position", "velocity", "affine", "deformation", "plastic"):
        assert np.array_equal(getattr(a, name), getattr(b, name)), name


@pytest.mark.parametrize("mode", ["fp32", "fixed64"])
def test_blocks_that_multiply_between_synchronizations(transfers, mode):
    rng = np.random.default_rng(3)
    pos = (16.6 + rng.uniform(0.0, 3.8, size=(900, 3))) * H
    vel = (pos - 18.5 * H) * 0.1 / DT  # one block expands to some hundred within the submission
    m = MaterialModel.fluid(1.0e-3, 7.0, 0.0)
    runs = []
    for steps in ((36,), (1,) * 36):
        s = HipMpmResidentSession(transfers, world_of(pos, vel, m), DT, mode)
        for k in steps:
            s.step(k)
        runs.append((s.read_particles(), s.topology_stats()))
        s.close()
    (a, ta), (b, tb) = runs
    assert ta == tb and ta["particle_blocks"] > 72  # 72: the grid launched for one block
    for name in ("position", "velocity", "affine", "deformation"):
        assert np.array_equal(getattr(a, name), getattr(b, name)), name


@pytest.mark.parametrize("graphs", ["0", "1"])
def test_launches_follow_full_binnings_without_a_synchronize(transfers, graphs, monkeypatch):
    # one block becomes hundreds over submissions that nothing waits for: the launch widths and
    # grids change on the way, the state does not
    rng = np.random.default_rng(3)
    pos = (16.6 + rng.uniform(0.0, 3.8, size=(3000, 3))) * H
    vel = (pos - 18.5 * H) * 0.1 / DT
    m = MaterialModel.fluid(1.0e-3, 7.0, 0.0)
    monkeypatch.setenv("TMPM_GRAPHS", graphs)
    runs = []
    for wait in (False, True):
        s = HipMpmResidentSession(transfers, world_of(pos, vel, m), DT, "fp32")
        for _ in range(34):
            s.submit_steps(3)
            if wait:
                s.synchronize()
        s.synchronize()
        runs.append((s.read_particles(), s.topology_stats()))
        s.close()
    (a, ta), (b, tb) = runs
    assert ta == tb and ta["particle_blocks"] > 512
    for name in ("position", "velocity", "affine", "deformation"):
        assert np.array_equal(getattr(a, name), getattr(b, name)), name
