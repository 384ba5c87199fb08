"""The rigid coupling of a substep in one launch (k_rigid_step) against its
three kernels, and over submissions of different lengths: the same bits."""

import numpy as np
import pytest

from tessera_amd.mpm import HipMpmBatch, HipMpmResidentSession, RigidMapping, RigidObstacle

from .test_gpu_coupling import box_on_slab

pytestmark = pytest.mark.gpu

G = np.array([0.0, -9.8, 0.0])
BODY = ("position", "orientation", "linear_velocity", "angular_velocity")


def crowded(seed, far):
    """The box on its slab and `far` spheres out of reach, some of them on the box's body."""
    w, bodies, maps = box_on_slab(seed)
    obstacles = list(w.obstacles) + [RigidObstacle.sphere([30.0 + 3.0 * i, 0.0, 0.0], 1.0) for i in range(far)]
    w.set_obstacles(obstacles)
    return w, bodies, maps + [RigidMapping(0, np.array([30.0 + 3.0 * i, 0.0, 0.0])) if i % 5 == 0 else RigidMapping(None)
                              for i in range(far)]


def same(a, b, obstacles_a, obstacles_b):
    for f in BODY:
        assert np.array_equal(getattr(a, f), getattr(b, f)), f
    for x, y in zip(obstacles_a, obstacles_b):
        for f in ("center", "orientation", "linear_velocity", "angular_velocity"):
            assert np.array_equal(getattr(x, f), getattr(y, f)), f


@pytest.mark.parametrize("far", [0, 90, 254])  # up to 1,536 components: one pass of the workgroup and several
def test_submissions_of_any_length_couple_the_same(transfers, far):
    w, bodies, maps = crowded(0, far)
    dt = min(5.0e-5, 0.5 * w.stable_timestep())
    runs = []
    for parts in ((12,), (1,) * 12, (5, 7)):
        s = HipMpmResidentSession(transfers, w, dt, "fixed64")
        s.set_rigid_bodies(bodies, maps, gravity=G, integrate=True)
        for k in parts:
            s.submit_steps(k)
        s.synchronize()
        runs.append((s.rigid_bodies()[0], s.obstacles(), s.reactions(), s.read_particles().position))
        s.close()
    for body, obstacles, reactions, position in runs[1:]:
        same(runs[0][0], body, runs[0][1], obstacles)
        assert np.array_equal(runs[0][2], reactions) and np.array_equal(runs[0][3], position)


def test_more_obstacles_than_one_workgroup_takes(transfers):
    scenes = [crowded(seed, 254) for seed in range(5)]  # 1,280 obstacles: the three kernels
    dt = min(5.0e-5, 0.5 * scenes[0][0].stable_timestep())
    batch = HipMpmBatch(transfers, [w for w, _, _ in scenes], [dt] * 5, "fixed64")
    for k, (_, bodies, maps) in enumerate(scenes):
        batch.set_rigid_bodies(k, bodies, maps, gravity=G)
    batch.step(9)
    for k in (0, 4):
        w, bodies, maps = scenes[k]
        alone = HipMpmResidentSession(transfers, w, dt, "fixed64")
        alone.set_rigid_bodies(bodies, maps, gravity=G)
        alone.step(9)
        same(alone.rigid_bodies()[0], batch.rigid_bodies(k)[0], alone.obstacles(), batch.obstacles(k))
        assert np.array_equal(alone.read_particles().position, batch.read_particles(k).position)
        alone.close()


def test_rigid_step_of_a_submission_over_reorders(transfers):
    # the rigid step rides on the next substep's list update except before a reorder and at the end
    w, bodies, maps = crowded(1, 3)
    dt = min(5.0e-5, 0.5 * w.stable_timestep())
    runs = []
    for parts in ((40,), (1,) * 40, (15, 2, 16, 7)):
        s = HipMpmResidentSession(transfers, w, dt, "fixed64")
        s.set_rigid_bodies(bodies, maps, gravity=G, integrate=True)
        for k in parts:
            s.submit_steps(k)
        s.synchronize()
        runs.append((s.rigid_bodies()[0], s.obstacles(), s.reactions(), s.read_particles().position))
        s.close()
    for body, obstacles, reactions, position in runs[1:]:
        same(runs[0][0], body, runs[0][1], obstacles)
        assert np.array_equal(runs[0][2], reactions) and np.array_equal(runs[0][3], position)
