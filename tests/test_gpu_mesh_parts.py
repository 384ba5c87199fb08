"""The winding test split over workgroups: the same candidates whatever part of
the split the allocation-free sampler's memory has room for, from one part up."""

import numpy as np
import pytest

from tessera_amd.mpm import HipMpmTransfers
from tests.test_zz_no_alloc import icosphere, sample

pytestmark = pytest.mark.gpu

SCRATCH = 32 << 20


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


# 320 triangles: at most 10 parts; about 30 to 8,000 candidates
@pytest.mark.parametrize("spacing", [0.2, 0.145, 0.031])
@pytest.mark.parametrize("room", [0.0, 1.0, 2.5, 9.9, 30.0])  # parts that fit, if one took 8 bytes a candidate
def test_parts_that_fit(transfers, spacing, room):
    v, t = icosphere(2)
    want = sample(False, transfers, v, t, spacing, 10**6, 10**5)
    count = int(np.prod(np.ceil((v.max(0) - v.min(0)) / spacing) + 1))
    left = 1024 + count + int(8 * count * room)
    spare = (SCRATCH - left - 12 * len(t) - 768) // 24 - len(v)
    padded = np.concatenate([v, np.tile(v[:1], (spare, 1))])  # vertices of no triangle
    assert len(want) and np.array_equal(sample(True, transfers, padded, t, spacing, 10**6, 10**5), want)
