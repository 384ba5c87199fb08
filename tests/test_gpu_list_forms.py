"""Listed substeps against a full binning of every substep, bit for bit, in the
forms of session that write lists by another kernel variant, with reorder
intervals beyond the lists' span, and in a batch that a scene drops out of."""

import numpy as np
import pytest

from tessera_amd.mpm import (HipMpmBatch, HipMpmResidentSession, HipMpmTransfers, MaterialModel, MpmParams, MpmWorld,
                             RigidObstacle, WorldBounds)
from tessera_amd.scenes import _particles

pytestmark = pytest.mark.gpu

H, DT = 1.0 / 64, 1.0e-4
FIELDS = ("position", "velocity", "affine", "deformation", "plastic")


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


def world(seed, material, obstacle=None, n=4000, speed=0.15):
    rng = np.random.default_rng(seed)
    pos = (20.6 + rng.uniform(0.0, 11.0, size=(n, 3))) * H
    vel = (np.array([1.0, -0.6, 0.4]) * speed + rng.normal(0.0, 0.02, size=pos.shape)) * H / DT
    pa = _particles(pos, vel, H / 4, 1.0e3, material)
    w = MpmWorld(pa, MpmParams(cell_width=H, gravity=np.array([0.0, -9.8, 0.0]), max_substep=DT, bounds=None))
    c = pos.mean(0) + np.array([0.12, -0.07, 0.05])
    if obstacle == "prism":
        w.set_obstacles([RigidObstacle.triangle_prism(c, [[0.0, -0.1, -0.1], [0.0, 0.1, -0.1], [0.0, 0.0, 0.1]], 0.02)])
    elif obstacle == "convex":
        corner = np.array([[x, y, z] for x in (-0.05, 0.05) for y in (-0.05, 0.05) for z in (-0.05, 0.05)])
        normals = [np.array(v, dtype=float) for v in ((1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1))]
        w.set_obstacles([RigidObstacle.convex(c, list(corner), normals)])
    return w


ELASTIC, SAND = MaterialModel.elastic(1.0e3, 0.3), MaterialModel.sand(1.0e3, 0.3, 0.6, 0.0)


def run(transfers, w, interval, react, monkeypatch):
    monkeypatch.setenv("TMPM_REORDER_INTERVAL", str(interval))
    s = HipMpmResidentSession(transfers, w, DT)
    if react:
        s.set_reactions(True)
    for k in (33, 64, 3):
        s.step(k)
    got = s.read_particles()
    s.close()
    return got


@pytest.mark.parametrize("material,obstacle,react", [(ELASTIC, None, False), (SAND, None, False), (ELASTIC, "prism", False),
                                                     (SAND, "prism", True), (ELASTIC, "convex", True)])
def test_listed_forms_equal_full_binning(transfers, material, obstacle, react, monkeypatch):
    w = world(1, material, obstacle)
    full = run(transfers, w, 1, react, monkeypatch)
    for interval in (16, 32, 33, 48):  # the last two end their lists within the interval
        got = run(transfers, w, interval, react, monkeypatch)
        for f in FIELDS:
            assert np.array_equal(getattr(got, f), getattr(full, f)), (interval, f)


def test_a_scene_that_drops_out_changes_no_other(transfers):
    worlds = [world(k, m) for k, m in ((1, ELASTIC), (2, SAND), (3, ELASTIC))]
    lo = worlds[1].particles.position.min(0)
    # the second scene leaves its grid within the 64 substeps
    worlds[1].params.bounds = WorldBounds(lo - 4 * H, worlds[1].particles.position.max(0) + 4 * H)
    worlds[1].particles.velocity[:] = np.array([0.35, 0.0, 0.0]) * H / DT
    worlds[1].params.gravity = np.zeros(3)
    b = HipMpmBatch(transfers, worlds, [DT] * 3, "fp32")
    b.submit_steps(64)
    b.synchronize()
    for k in (0, 2):
        s = HipMpmResidentSession(transfers, worlds[k], DT)
        s.step(64)
        alone, got = s.read_particles(), b.read_particles(k)
        assert b.scene_error(k) is None and b.substeps(k) == 64
        for f in FIELDS:
            assert np.array_equal(getattr(got, f), getattr(alone, f)), (k, f)
        s.close()
    b.close()
