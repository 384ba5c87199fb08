"""What a user of the MLS-MPM backend has it do, as cases that can be timed.

Every case is one call (or the few calls of one frame) through the public
entry points of ``tessera_amd``:

``frame``     a resident session: some fixed substeps are submitted and the
              particle snapshot is encoded into a device buffer, as a renderer
              or a learning loop on the device does each frame.  One scene of
              any size, in either P2G mode.
``batch``     many uneven scenes advanced together, then the snapshot.
``serving``   one tick of the serving loop: scenes with falling rigid boxes
              coupled to the particles, reactions on, then the snapshot and
              the bodies' poses.
``readback``  a resident session is stepped and its whole particle state is
              read back to the host (a simulation whose host side looks at
              every frame).
``adaptive``  the CFL-limited step of the ``MpmWorld`` API, then the readback.
``fill``      a closed triangle mesh is filled with particles (mesh emitter).

Sizes run from 500 particles and one substep to the 4,194,304-particle dam
break; most are odd or ragged.  Velocities are not zero, as in a scene that
is under way, and the scenes are bounded, so they can be stepped for long.
"""

from __future__ import annotations

import math

import numpy as np
import torch

GRAVITY = (0.0, -9.8, 0.0)
DAM_CELL = 0.0048559


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # A control or editing loop: few particles, one substep a call, where launches and latency count.
        dict(name="cube_2k_one_substep", kind="frame", scene="cube", material="elastic", n=1999, cells=64, dt=1e-4,
             substeps=1, mode="fp32"),
        # The 8,192-particle cube on a sticky floor (C1), a frame of 20 substeps.
        dict(name="cube_8k_frame", kind="frame", scene="cube", material="elastic", n=8192, cells=64, dt=1e-4,
             substeps=20, mode="fp32"),
        # Plastic flow: a sand heap of middling, ragged size on the floor.
        dict(name="sand_79k_frame", kind="frame", scene="cube", material="sand", n=79507, cells=96, dt=1e-4, substeps=10,
             mode="fp32"),
        # The headline scene (C2): 1,048,576 elastic particles in four cubes.
        dict(name="four_cubes_1m_frame", kind="frame", scene="four_cubes", material="elastic", n=1048576, cells=256,
             dt=5e-5, substeps=10, mode="fp32"),
        # The reproducible fixed-point mode, at a ragged size.
        dict(name="four_cubes_415k_fixed64", kind="frame", scene="four_cubes", material="elastic", n=415292, cells=192,
             dt=5e-5, substeps=10, mode="fixed64"),
        # The largest scene (C3): a 4,194,304-particle fluid column in flow.
        dict(name="dam_break_4m_frame", kind="frame", scene="dam", material="fluid", n=4194304, cells=206, dt=2e-5,
             substeps=6, mode="fp32"),
        # Uneven scenes as one batch (C4's distribution: 2,048 to 65,536 particles each, mixed materials).
        dict(name="batch_128_scenes", kind="batch", scenes=128, n_min=2048, n_max=65536, substeps=16, mode="fp32"),
        # A few tiny scenes as one batch: a small parameter sweep.
        dict(name="batch_9_small_scenes", kind="batch", scenes=9, n_min=500, n_max=4000, substeps=16, mode="fp32"),
        # One serving tick (C5's distribution: 4,096 to 524,288 particles, 1-4 rigid boxes, 32 substeps a tick).
        dict(name="serving_tick_16_scenes", kind="serving", scenes=16, n_min=4096, n_max=524288, substeps=32,
             mode="fp32"),
        # A host program that reads every frame back.
        dict(name="readback_59k", kind="readback", scene="cube", material="neo_hookean", n=59319, cells=128, dt=5e-5,
             substeps=10, mode="fp32"),
        # The CFL-limited step with its per-substep validation, small scene.
        dict(name="adaptive_4k", kind="adaptive", scene="cube", material="elastic", n=4097, cells=64, dt=1e-4, substeps=8,
             mode="fp32"),
        # Mesh emission: an icosphere of 1,280 triangles over about 50,000 lattice candidates.
        dict(name="fill_mesh_1280", kind="fill", level=3, spacing=0.0271, radius=0.4),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "batch", "serving", "readback", "adaptive", "fill"])
    mode = rng.choice(["fp32", "fp32", "fp32", "fixed64"])
    if kind == "frame":
        scene = rng.choice(["cube", "cube", "four_cubes", "dam"])
        n = _log_uniform(rng, 500, 2000000) | 1
        material = "fluid" if scene == "dam" else rng.choice(["elastic", "neo_hookean", "fluid", "sand"])
        if material == "sand":
            n = min(n, 150001)
        return dict(kind=kind, scene=scene, material=material, n=n, cells=_cells(scene, n), dt=_dt(scene, n),
                    substeps=_substeps(rng, n), mode=mode)
    if kind == "batch":
        lo = _log_uniform(rng, 300, 4000)
        return dict(kind=kind, scenes=rng.randrange(2, 97), n_min=lo, n_max=lo * rng.randrange(2, 17),
                    substeps=rng.randrange(4, 33), mode=mode)
    if kind == "serving":
        lo = _log_uniform(rng, 2048, 8192)
        return dict(kind=kind, scenes=rng.randrange(1, 17), n_min=lo, n_max=lo * rng.randrange(2, 41),
                    substeps=rng.randrange(8, 33), mode=mode)
    if kind == "fill":
        level = rng.randrange(1, 4)
        return dict(kind=kind, level=level, spacing=round(rng.uniform(0.022, 0.06), 5), radius=round(rng.uniform(0.2, 0.4), 4))
    n = _log_uniform(rng, 500, 100000 if kind == "readback" else 10000) | 1
    return dict(kind=kind, scene="cube", material=rng.choice(["elastic", "neo_hookean", "fluid"]), n=n,
                cells=_cells("cube", n), dt=_dt("cube", n), substeps=rng.randrange(2, 13), mode=mode)


def _cells(scene, n):
    """Cells per metre that give about the density of the configured scenes (2 to 10 particles a cell)."""
    if scene == "dam":
        return max(16, min(256, int(round((n / (0.24 * 2.0)) ** (1.0 / 3.0)))))
    if scene == "four_cubes":
        return max(32, min(256, int(round((n / (0.032 * 2.0)) ** (1.0 / 3.0)))))
    return max(32, min(192, int(round((n / (0.064 * 6.0)) ** (1.0 / 3.0)))))


def _dt(scene, n):
    c = _cells(scene, n)
    return 1e-4 if c <= 64 else 5e-5 if c <= 192 else 2e-5


def _substeps(rng, n):
    return rng.randrange(1, 33) if n < 100000 else rng.randrange(2, 13)


# ---------------------------------------------------------------------------
# Scenes.  Positions, velocities and per-particle scalars are FP32 values (what
# the device holds), in the FP64 arrays of the API.
# ---------------------------------------------------------------------------
def _f32(a):
    return np.asarray(a, dtype=np.float32).astype(np.float64)


MATERIALS = ("elastic", "neo_hookean", "fluid", "sand")
YOUNG, POISSON, FRICTION = 1.0e4, 0.3, math.radians(35.0)
BULK, GAMMA = 1.0e5, 7.0


def _material(name):
    from tessera_amd.mpm import MaterialModel

    if name == "elastic":
        return MaterialModel.elastic(YOUNG, POISSON)
    if name == "neo_hookean":
        return MaterialModel.neo_hookean(YOUNG, POISSON)
    if name == "fluid":
        return MaterialModel.fluid(BULK, GAMMA, 0.0)
    return MaterialModel.sand(YOUNG, POISSON, FRICTION, 0.0)


def _jittered_box(rng, n, lo, hi):
    """n points of a jittered lattice over the box, the last layers left out where n is no full lattice."""
    lo, hi = np.asarray(lo, float), np.asarray(hi, float)
    ext = hi - lo
    s = (float(np.prod(ext)) / n) ** (1.0 / 3.0)
    counts = np.maximum(1, np.ceil(ext / s - 1e-9).astype(int))
    while counts.prod() < n:
        counts[int(np.argmax(ext / counts))] += 1
    i = np.arange(n)
    idx = np.stack([i // (counts[1] * counts[2]), (i // counts[2]) % counts[1], i % counts[2]], axis=1)
    return lo + (idx + rng.random((n, 3), dtype=np.float32)) * (ext / counts)


def _flow(rng, pos, noise, shear):
    """A velocity field under way: a shear flow and noise."""
    v = rng.standard_normal(pos.shape, dtype=np.float32) * noise
    v[:, 0] += shear * (pos[:, 1] - 0.5)
    v[:, 2] -= shear * (pos[:, 0] - 0.5)
    return v


def _scene_arrays(case, seed):
    """(positions, velocities, rest volume, density, cell width) of a single scene."""
    rng = np.random.default_rng([seed, case["n"]])
    n = case["n"]
    if case["scene"] == "dam":
        h = DAM_CELL if n == 4194304 else 1.0 / (case["cells"] + 0.37)
        pos = _jittered_box(rng, n, [0.0, 0.0, 0.0], [0.4, 0.6, 1.0])
        volume = 0.24 / n
        vel = _flow(rng, pos, 0.2, 0.4)
    elif case["scene"] == "four_cubes":
        h = 1.0 / case["cells"]
        centers = np.array([[0.3, 0.3, 0.3], [0.7, 0.3, 0.7], [0.3, 0.7, 0.7], [0.7, 0.7, 0.3]])
        sizes = [n // 4 + (k < n % 4) for k in range(4)]
        pos = np.concatenate([_jittered_box(rng, m, c - 0.1, c + 0.1) for m, c in zip(sizes, centers) if m])
        volume = 0.032 / n
        vel = rng.standard_normal(pos.shape, dtype=np.float32) * np.float32(0.5)
    else:
        h = 1.0 / case["cells"]
        edge = 0.2 if n <= 8192 else 0.4
        lo = np.array([0.5 - edge / 2, 0.06, 0.5 - edge / 2])
        pos = _jittered_box(rng, n, lo, lo + edge)
        volume = edge ** 3 / n
        vel = _flow(rng, pos, 0.2, 1.0)
    return _f32(pos), _f32(vel), float(np.float32(volume)), 1000.0, h


def _world(pos, vel, volume, density, h, material, dt, floor):
    from tessera_amd.mpm import MpmParams, MpmWorld, ParticleArrays, WorldBounds
    from tessera_amd.scenes import sticky_floor

    m = _material(material)
    pa = ParticleArrays(len(pos), [m])
    pa.position[:] = pos
    pa.velocity[:] = vel
    pa.rest_volume[:] = volume
    pa.mass[:] = np.float32(density * volume)
    pa.radius[:] = 0.5 * volume ** (1.0 / 3.0)
    if material == "sand":
        pa.plastic[:, 1] = 1.0
    params = MpmParams(cell_width=h, gravity=np.array(GRAVITY), max_substep=dt,
                       bounds=WorldBounds(np.zeros(3), np.ones(3)))
    w = MpmWorld(pa, params)
    if floor:
        w.set_obstacles([sticky_floor(0.05)])
    return w


def _batch_arrays(case, seed):
    """Per scene: (positions, velocities, rest volume, density, cell width, material)."""
    rng = np.random.default_rng([seed, case["scenes"]])
    out = []
    # the scenes' sizes spread evenly over the logarithm, so that the work does not vary with the seed
    for k in range(case["scenes"]):
        n = int(round(case["n_min"] * (case["n_max"] / case["n_min"]) ** ((k + 0.5) / case["scenes"])))
        h = 1.0 / (64, 80, 96, 112, 128)[k % 5]
        edge = (n / 8.0) ** (1.0 / 3.0) * h
        lo = rng.uniform(0.2, 0.8 - edge, size=3)
        pos = _jittered_box(rng, n, lo, lo + edge)
        vel = rng.standard_normal(pos.shape, dtype=np.float32) * np.float32(0.3)
        out.append((_f32(pos), _f32(vel), float(np.float32(h ** 3 / 8.0)), 1000.0, h, MATERIALS[k % 3]))
    return out


MAX_BOXES = 4


def _serving_requests(case, seed):
    from tessera_amd.scenes import serving_request

    rng = np.random.default_rng([seed, case["scenes"], 5])
    out = []
    for k in range(case["scenes"]):
        n = int(round(case["n_min"] * (case["n_max"] / case["n_min"]) ** ((k + 0.5) / case["scenes"])))
        out.append(serving_request(rng, n, "request %d" % k, 2000, 0.0, MAX_BOXES))
    return out


def _icosphere(level, radius, center):
    t = (1.0 + math.sqrt(5.0)) / 2.0
    v = [np.array(p, float) / math.sqrt(1.0 + t * t) for p in
         [(-1, t, 0), (1, t, 0), (-1, -t, 0), (1, -t, 0), (0, -1, t), (0, 1, t), (0, -1, -t), (0, 1, -t),
          (t, 0, -1), (t, 0, 1), (-t, 0, -1), (-t, 0, 1)]]
    f = [(0, 11, 5), (0, 5, 1), (0, 1, 7), (0, 7, 10), (0, 10, 11), (1, 5, 9), (5, 11, 4), (11, 10, 2), (10, 7, 6),
         (7, 1, 8), (3, 9, 4), (3, 4, 2), (3, 2, 6), (3, 6, 8), (3, 8, 9), (4, 9, 5), (2, 4, 11), (6, 2, 10), (8, 6, 7),
         (9, 8, 1)]
    for _ in range(level):
        mid, nf = {}, []

        def m(a, b):
            k = (min(a, b), max(a, b))
            if k not in mid:
                p = v[a] + v[b]
                v.append(p / np.linalg.norm(p))
                mid[k] = len(v) - 1
            return mid[k]

        for a, b, c in f:
            ab, bc, ca = m(a, b), m(b, c), m(c, a)
            nf += [(a, ab, ca), (b, bc, ab), (c, ca, bc), (ab, bc, ca)]
        f = nf
    return np.array(v) * radius + np.asarray(center), np.array(f, dtype=np.uint32)


def _mesh(case, seed):
    """An uneven, turned icosphere, the case's own, at a place and with triangles in an order of the seed's
    (the lattice is laid from the mesh's own corner, so the number of samples is the case's)."""
    rng = np.random.default_rng(case["level"])
    v, f = _icosphere(case["level"], 1.0, np.zeros(3))
    q, r = np.linalg.qr(rng.standard_normal((3, 3)))
    q = q * np.sign(np.diag(r))
    if np.linalg.det(q) < 0:
        q[:, 0] = -q[:, 0]
    axes = case["radius"] * rng.uniform(0.8, 1.0, size=3)
    place = np.random.default_rng([seed, case["level"]])
    return (v * axes) @ q.T + place.uniform(0.45, 0.55, size=3), f[place.permutation(len(f))]


# ---------------------------------------------------------------------------
# What a program has in hand, and the pass
# ---------------------------------------------------------------------------
_TRANSFERS = []


def _transfers():
    from tessera_amd.mpm import HipMpmTransfers

    if not _TRANSFERS:
        _TRANSFERS.append(HipMpmTransfers(0))
    return _TRANSFERS[0]


def prepare(case, seed):
    from tessera_amd.mpm import HipMpmBatch, HipMpmResidentSession

    t = _transfers()
    kind = case["kind"]
    state = dict(case=case, transfers=t)
    if kind == "fill":
        from tessera_amd.emitters import MeshEmitter

        v, f = _mesh(case, seed)
        state["emitter"] = MeshEmitter(v, f, case["spacing"], 1000.0, _material("elastic"), 1 << 20, 1 << 18)
        return state
    if kind == "batch":
        scenes = _batch_arrays(case, seed)
        worlds = [_world(p, v, vol, rho, h, m, 5e-5, False) for p, v, vol, rho, h, m in scenes]
        state["session"] = HipMpmBatch(t, worlds, [5e-5] * len(worlds), case["mode"])
        n = sum(len(w.particles) for w in worlds)
    elif kind == "serving":
        reqs = _serving_requests(case, seed)
        b = HipMpmBatch(t, [r.world for r in reqs], [r.dt for r in reqs], case["mode"])
        b.set_reactions(True)
        for k, r in enumerate(reqs):
            b.set_rigid_bodies(k, r.bodies, r.mappings, gravity=GRAVITY)
        state["session"] = b
        n = sum(len(r.world.particles) for r in reqs)
    else:
        pos, vel, vol, rho, h = _scene_arrays(case, seed)
        w = _world(pos, vel, vol, rho, h, case["material"], case["dt"], case["scene"] == "cube")
        state["session"] = HipMpmResidentSession(t, w, case["dt"], case["mode"])
        n = len(pos)
    if kind in ("frame", "batch", "serving"):
        state["snapshot"] = torch.zeros((n, 8), dtype=torch.float32, device="cuda")
    return state


def run(state):
    from tessera_amd.mpm import HipMpmResidentSession

    case = state["case"]
    kind = case["kind"]
    if kind == "fill":
        p = state["emitter"].sample(state["transfers"])
        return {"position": p.position, "mass": p.mass}
    s = state["session"]
    k = case["substeps"]
    if kind in ("readback", "adaptive"):
        if kind == "readback":
            s.step(k)
        else:
            s.step_adaptive(k * case["dt"])
        p = s.read_particles()
        # the device state is FP32 and the readback widens it: kept as FP32 columns
        return {f: np.asarray(getattr(p, f), dtype=np.float32) for f in
                ("position", "velocity", "deformation", "affine", "mass")}
    if kind == "frame":
        s.submit_steps(k)
    else:
        s.step(k)
    buf = state["snapshot"]
    # the same session-level entry point for sessions and batches
    HipMpmResidentSession.encode_particle_snapshot(s, buf.data_ptr(), buf.numel() * 4)
    out = {"position_mass": buf[:, :4], "velocity_volume": buf[:, 4:]}
    if kind == "serving":
        poses = np.zeros((case["scenes"], MAX_BOXES, 2, 3), dtype=np.float32)
        for scene in s.scenes():
            for b, body in enumerate(s.rigid_bodies(scene)):
                poses[scene, b] = body.position, body.linear_velocity
        out["bodies"] = poses
    return out


# Per particle and substep: the state is read once and written once (x, v, C, F; mass and volume read), and
# P2G and G2P each visit 27 nodes (a weight, and for P2G four, for G2P three accumulations with an affine
# term: about 600 operations each), with some 200 for the stress.
BYTES_PARTICLE, FLOPS_PARTICLE = 200, 1400


def work(case):
    kind = case["kind"]
    if kind == "fill":
        tris = 20 * 4 ** case["level"]
        candidates = (2.0 * case["radius"] / case["spacing"]) ** 3
        return {"bytes": 24.0 * candidates * 0.52, "flops": 60.0 * tris * candidates}
    if kind in ("batch", "serving"):
        n = sum(int(round(case["n_min"] * (case["n_max"] / case["n_min"]) ** ((k + 0.5) / case["scenes"])))
                for k in range(case["scenes"]))
    else:
        n = case["n"]
    out = 200.0 if kind in ("readback", "adaptive") else 32.0
    return {"bytes": float(n) * (BYTES_PARTICLE * case["substeps"] + out),
            "flops": float(n) * FLOPS_PARTICLE * case["substeps"]}


# ---------------------------------------------------------------------------
# The same in 64 bits, with plain torch
# ---------------------------------------------------------------------------
def _cofactors(F):
    a, b, c = F[:, :, 0], F[:, :, 1], F[:, :, 2]
    cross = torch.linalg.cross
    return torch.stack([cross(b, c), cross(c, a), cross(a, b)], dim=2), (a * cross(b, c)).sum(1)


def _det(F):
    return _cofactors(F)[1]


def _product(A, B):
    return (A[:, :, :, None] * B[:, None, :, :]).sum(2)


def _polar(F):
    R = F
    for _ in range(10):
        cof, det = _cofactors(R)
        R = 0.5 * (R + cof / det[:, None, None])
    return R


def _kirchhoff(material, F):
    lam = YOUNG * POISSON / ((1.0 + POISSON) * (1.0 - 2.0 * POISSON))
    mu = YOUNG / (2.0 * (1.0 + POISSON))
    eye = torch.eye(3, dtype=F.dtype, device=F.device)
    J = _det(F)
    if material == "neo_hookean":
        return mu * _product(F, F.transpose(1, 2)) + (lam * torch.log(J.clamp_min(1e-10)) - mu)[:, None, None] * eye
    if material == "fluid":
        sj = J.clamp_min(1e-6)
        p = torch.where(sj <= 1.0, BULK * (sj ** -GAMMA - 1.0), -BULK * 0.25 * (sj - 1.0))
        return (-p * sj)[:, None, None] * eye
    R = _polar(F)
    return 2.0 * mu * _product(F - R, F.transpose(1, 2)) + (lam * (J - 1.0) * J)[:, None, None] * eye


def _project_sand(F, plastic):
    """Drucker-Prager return mapping with friction hardening; plastic: (n, 3) det, hardening, log volume gain."""
    lam = YOUNG * POISSON / ((1.0 + POISSON) * (1.0 - 2.0 * POISSON))
    mu = YOUNG / (2.0 * (1.0 + POISSON))
    w, V = torch.linalg.eigh(_product(F.transpose(1, 2), F).cpu())
    w, V = w.to(F.device), V.to(F.device)
    s = w.clamp_min(1e-24).sqrt()
    strain = s.log() + plastic[:, 2:3] / 3.0
    tr = strain.sum(1, keepdim=True)
    dev = strain - tr / 3.0
    norm = dev.norm(dim=1, keepdim=True)
    q = plastic[:, 1:2]
    deg = math.pi / 180.0
    sine = torch.sin(FRICTION + (9.0 * deg * q - 10.0 * deg) * torch.exp(-0.2 * q))
    alpha = math.sqrt(2.0 / 3.0) * 2.0 * sine / (3.0 - sine)
    tension = (tr > 0.0) | (norm <= 4.76837158203125e-7)
    gamma = norm + (3.0 * lam + 2.0 * mu) / (2.0 * mu) * tr * alpha
    inside = ~tension & (gamma <= 0.0)
    logs = torch.where(tension, torch.zeros_like(strain), strain - dev * (gamma / norm.clamp_min(1e-300)))
    inc = torch.where(tension, strain.norm(dim=1, keepdim=True), gamma)
    out = logs.exp()
    scale = torch.where(inside, torch.ones_like(out), out / s)
    Fn = _product(F, _product(V * scale[:, None, :], V.transpose(1, 2)))
    old, new = s.prod(1, keepdim=True), out.prod(1, keepdim=True)
    moved = torch.cat([(plastic[:, 0:1] * old / new).clamp(0.01, 100.0), plastic[:, 1:2] + inc,
                       plastic[:, 2:3] + old.log() - new.log()], dim=1)
    return torch.where(inside[:, :, None], F, Fn), torch.where(inside, plastic, moved)


def _advance(pos, vel, volume, density, h, material, dt, substeps, floor):
    """x, v, F, C after the substeps, all in 64 bits."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x = torch.tensor(pos, dtype=torch.float64, device=dev)
    v = torch.tensor(vel, dtype=torch.float64, device=dev)
    n = len(x)
    F = torch.eye(3, dtype=torch.float64, device=dev).repeat(n, 1, 1)
    Cm = torch.zeros((n, 3, 3), dtype=torch.float64, device=dev)
    plastic = torch.tensor([1.0, 1.0, 0.0], dtype=torch.float64, device=dev).repeat(n, 1)
    mass = float(np.float32(density * volume))
    radius = 0.5 * volume ** (1.0 / 3.0)
    g = torch.tensor(GRAVITY, dtype=torch.float64, device=dev)
    inv_d = 4.0 / (h * h)
    for _ in range(substeps):
        base = torch.floor(x / h - 0.5).to(torch.int64)
        fx = x / h - base
        w = torch.stack([0.5 * (1.5 - fx) ** 2, 0.75 - (fx - 1.0) ** 2, 0.5 * (fx - 0.5) ** 2])
        origin = base.min(dim=0).values
        dims = (base.max(dim=0).values - origin + 3).tolist()
        flat = ((base - origin)[:, 0] * dims[1] + (base - origin)[:, 1]) * dims[2] + (base - origin)[:, 2]
        A = mass * Cm - (dt * volume * inv_d) * _kirchhoff(material, F)
        grid = torch.zeros((dims[0] * dims[1] * dims[2], 4), dtype=torch.float64, device=dev)
        nodes = [(a, b, c) for a in range(3) for b in range(3) for c in range(3)]
        for a, b, c in nodes:
            wt = w[a, :, 0] * w[b, :, 1] * w[c, :, 2]
            d = (torch.tensor([a, b, c], dtype=torch.float64, device=dev) - fx) * h
            p = mass * v + (A * d[:, None, :]).sum(2)
            grid.index_add_(0, flat + (a * dims[1] + b) * dims[2] + c,
                            torch.cat([(wt * mass)[:, None], wt[:, None] * p], dim=1))
        live = grid[:, 0] > 0.0
        gv = torch.where(live[:, None], grid[:, 1:] / torch.where(live, grid[:, 0], 1.0)[:, None] + g * dt, 0.0)
        i = torch.arange(len(grid), device=dev)
        ijk = torch.stack([i // (dims[1] * dims[2]), (i // dims[2]) % dims[1], i % dims[2]], dim=1) + origin
        np_ = ijk.to(torch.float64) * h
        eps = 1e-6 * h
        stop = ((np_ <= h + eps) & (gv < 0.0)) | ((np_ >= 1.0 - h - eps) & (gv > 0.0))
        gv = torch.where(stop, 0.0, gv)
        if floor:
            gv = torch.where((np_[:, 1:2] - 0.05 <= h * (1.0 + 1e-5)), 0.0, gv)
        v = torch.zeros_like(v)
        Cm = torch.zeros_like(Cm)
        for a, b, c in nodes:
            wt = w[a, :, 0] * w[b, :, 1] * w[c, :, 2]
            d = (torch.tensor([a, b, c], dtype=torch.float64, device=dev) - fx) * h
            nv = gv[flat + (a * dims[1] + b) * dims[2] + c] * wt[:, None]
            v = v + nv
            Cm = Cm + nv[:, :, None] * (d * inv_d)[:, None, :]
        x = x + v * dt
        low, high = x < radius, x > 1.0 - radius
        x = x.clamp(radius, 1.0 - radius)
        v = torch.where(low, v.clamp_min(0.0), torch.where(high, v.clamp_max(0.0), v))
        if floor:
            hit = x[:, 1:2] - 0.05 < radius
            x = torch.cat([x[:, 0:1], torch.where(hit, 0.05 + radius, x[:, 1:2]), x[:, 2:3]], dim=1)
            v = torch.where(hit, 0.0, v)
        F = F + dt * _product(Cm, F)
        if material == "fluid":
            s = _det(F).clamp_min(1e-9) ** (1.0 / 3.0)
            F = s[:, None, None] * torch.eye(3, dtype=torch.float64, device=dev)
        elif material == "sand":
            F, plastic = _project_sand(F, plastic)
    return x, v, F, Cm, mass


def _snapshot64(x, v, volume, mass):
    one = torch.ones((len(x), 1), dtype=torch.float64, device=x.device)
    return {"position_mass": torch.cat([x, mass * one], dim=1), "velocity_volume": torch.cat([v, volume * one], dim=1)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "serving":
        return None  # coupled rigid bodies: no plain restatement
    if kind == "fill":
        # the lattice centres inside the mesh, from the solid angles the triangles span
        v, f = _mesh(case, seed)
        lo, hi = v.min(axis=0), v.max(axis=0)
        sp = case["spacing"]
        counts = [int(math.ceil((b - a) / sp)) for a, b in zip(lo, hi)]
        i = np.stack(np.meshgrid(*[np.arange(c) for c in counts], indexing="ij"), axis=-1).reshape(-1, 3)
        p = lo + (i + 0.5) * sp
        p = torch.tensor(p[np.all(p < hi, axis=1)])
        tri = torch.tensor(v[f.astype(np.int64)])
        inside = []
        for c in p.split(4096):
            a, b, d = (tri[None, :, k, :] - c[:, None, :] for k in range(3))
            la, lb, ld = a.norm(dim=2), b.norm(dim=2), d.norm(dim=2)
            num = (a * torch.linalg.cross(b, d)).sum(2)
            den = la * lb * ld + (a * b).sum(2) * ld + (b * d).sum(2) * la + (d * a).sum(2) * lb
            inside.append((2.0 * torch.atan2(num, den)).sum(1).abs() > 2.0 * math.pi)
        p = p[torch.cat(inside)].numpy()
        return {"position": p, "mass": np.full(len(p), 1000.0 * sp ** 3)}
    if kind == "batch":
        parts = []
        for p, v, vol, rho, h, m in _batch_arrays(case, seed):
            x, w, _, _, mass = _advance(p, v, vol, rho, h, m, 5e-5, case["substeps"], False)
            parts.append(_snapshot64(x, w, vol, mass))
        return {f: torch.cat([q[f] for q in parts]) for f in ("position_mass", "velocity_volume")}
    pos, vel, vol, rho, h = _scene_arrays(case, seed)
    x, v, F, Cm, mass = _advance(pos, vel, vol, rho, h, case["material"], case["dt"], case["substeps"],
                                 case["scene"] == "cube")
    if kind == "frame":
        return _snapshot64(x, v, vol, mass)
    return {"position": x, "velocity": v, "deformation": F, "affine": Cm,
            "mass": torch.full((len(x),), mass, dtype=torch.float64)}
