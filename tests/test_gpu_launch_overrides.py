"""Launch widths set in the environment: reported as they run, and every kernel
that they select computes the same state bit for bit."""

import numpy as np
import pytest

from tessera_amd.mpm import (HipMpmResidentSession, HipMpmTransfers, MaterialModel, MpmParams, MpmWorld,
                             RigidObstacle)
from tessera_amd.scenes import _particles

pytestmark = pytest.mark.gpu

H, DT = 1.0 / 64, 1.0e-4


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


def world(material, prism):
    rng = np.random.default_rng(9)
    pos = (16.6 + rng.uniform(0.0, 22.0, size=(9000, 3))) * H
    pa = _particles(pos, rng.normal(0.0, 0.02 * H / DT, size=pos.shape), H / 4, 1.0e3, material)
    w = MpmWorld(pa, MpmParams(cell_width=H, gravity=np.array([0.0, -9.8, 0.0]), max_substep=DT, bounds=None))
    if prism:
        w.set_obstacles([RigidObstacle.triangle_prism(pos.mean(0), [[0.0, -0.1, -0.1], [0.0, 0.1, -0.1],
                                                                    [0.0, 0.0, 0.1]], 0.02)])
    return w


ELASTIC, SAND = MaterialModel.elastic(1.0e4, 0.3), MaterialModel.sand(1.0e4, 0.3, 0.6, 0.0)


@pytest.mark.parametrize("mode", ["fp32", "fixed64"])
@pytest.mark.parametrize("material,prism,p2g,g2p", [
    (ELASTIC, False, (64, 128, 256, 512), (64, 128, 256, 512)),
    (ELASTIC, True, (64, 128, 256, 512), (64, 128, 256, 256)),   # no G2P of 512 with shapes
    (SAND, False, (128, 128, 256, 512), (64, 128, 256, 256)),    # nor plastic, and no P2G of 64
])
def test_overrides_run_as_reported(transfers, material, prism, p2g, g2p, mode, monkeypatch):
    w = world(material, prism)
    monkeypatch.setenv("TMPM_P2G_COPIES", "1")
    runs = []
    for k, width in enumerate((64, 128, 256, 512)):
        monkeypatch.setenv("TMPM_P2G_THREADS", str(width))
        monkeypatch.setenv("TMPM_PBLOCK_THREADS", str(width))
        s = HipMpmResidentSession(transfers, w, DT, mode)
        cfg = s.launch_config()
        assert (cfg["p2g_threads"], cfg["p2g_copies"], cfg["g2p_threads"]) == (p2g[k], 1, g2p[k])
        s.step(19)
        runs.append(s.read_particles())
        s.close()
    for got in runs[1:]:
        for f in ("position", "velocity", "affine", "deformation", "plastic"):
            assert np.array_equal(getattr(got, f), getattr(runs[0], f)), f
