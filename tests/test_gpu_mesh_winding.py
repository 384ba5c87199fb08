"""The mesh sampler's winding test (k_mesh_winding) against the sum of the
triangles' solid angles in numpy, at the sizes where its split can go wrong."""

import numpy as np
import pytest

from tessera_amd.emitters import sample_closed_mesh_volume
from tessera_amd.mpm import HipMpmTransfers
from tests.test_zz_no_alloc import CUBE_T, CUBE_V, icosphere, sample

pytestmark = pytest.mark.gpu

TET_V = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], float)
TET_T = np.array([[0, 2, 1], [0, 1, 3], [0, 3, 2], [1, 2, 3]], np.uint32)


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


def inside(v, t, p):
    """|solid angle| > 2 pi, and the least distance of any triangle's number from the negative real axis."""
    a, b, c = (v[t[:, k]][None] - p[:, None] for k in range(3))
    la, lb, lc = (np.linalg.norm(q, axis=2) for q in (a, b, c))
    num = np.einsum("ijk,ijk->ij", a, np.cross(b, c))
    dot = lambda q, r: np.einsum("ijk,ijk->ij", q, r)
    den = la * lb * lc + dot(a, b) * lc + dot(b, c) * la + dot(c, a) * lb
    clear = np.where(den > 0, np.hypot(num, den), np.abs(num)) / (la * lb * lc)
    return np.abs(2.0 * np.arctan2(num, den).sum(1)) > 2.0 * np.pi, clear.min(1)


def overlapping(levels):
    v, t = icosphere(levels)
    return np.concatenate([v, v + [0.2, 0.05, 0.0]]), np.concatenate([t, t + len(v)])


MESHES = {
    "tetrahedron": (TET_V, TET_T, (0.9, 0.24, 0.05)),
    "cube": (CUBE_V, CUBE_T, (0.25, 0.2501, 0.063)),
    "reversed": (CUBE_V * 3.0 - 7.0, CUBE_T[:, ::-1], (0.41,)),
    "icosphere_80": (*icosphere(1), (0.6, 0.15, 0.021)),
    "icosphere_5120": (*icosphere(4), (0.11, 0.06)),
    "overlapping": (*overlapping(2), (0.053,)),
    "small_scale": (CUBE_V * 1e-3, CUBE_T, (1.7e-4,)),
}


@pytest.mark.parametrize("name", sorted(MESHES))
def test_winding_equals_the_sum_of_solid_angles(transfers, name):
    v, t, spacings = MESHES[name]
    t = np.ascontiguousarray(t)
    for spacing in spacings:
        lo, hi = v.min(0), v.max(0)
        counts = np.ceil((hi - lo) / spacing).astype(int)
        grid = np.stack(np.meshgrid(*[np.arange(c) for c in counts], indexing="ij"), -1).reshape(-1, 3)
        pts = lo + (grid + 0.5) * spacing
        pts = pts[np.all(pts < hi, axis=1)]
        parts = [inside(v, t, p) for p in np.array_split(pts, max(1, len(pts) * len(t) // 2_000_000))]
        want, clear = (np.concatenate([q[k] for q in parts]) for k in range(2))
        got = sample_closed_mesh_volume(transfers, v, t, spacing, 10**7, 10**6)
        # on the surface itself rounding decides; everywhere else both agree
        settled = clear > 1e-12
        assert settled.mean() > 0.5
        got_set = {tuple(p) for p in got}
        for p, w, s in zip(pts, want, settled):
            assert not s or (tuple(p) in got_set) == w, (spacing, p)
        assert np.array_equal(got, sample(True, transfers, v, t, spacing, 10**7, 10**6))
