"""Block lists that an edit takes away before any substep ran on them are not
made again at every substep."""

import numpy as np
import pytest

from tessera_amd.mpm import HipMpmBatch, HipMpmTransfers, StagedScene
from tests.test_gpu_batch import dts_for, mixed_worlds

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def transfers():
    return HipMpmTransfers(0)


@pytest.mark.parametrize("steps", [1, 2])
def test_admissions_between_substeps(transfers, steps, monkeypatch):
    worlds = mixed_worlds()[:3]
    dts = dts_for(worlds)
    runs = []
    for interval in ("1", "16"):
        monkeypatch.setenv("TMPM_REORDER_INTERVAL", interval)
        b = HipMpmBatch(transfers, worlds[:2], dts[:2], "fp32")
        b.set_timing(True)
        extra = None
        for _ in range(48):
            slot = b.add_staged(StagedScene(worlds[2], dts[2]))
            if extra is not None:
                b.remove_scene(extra)
            extra = slot
            b.step(steps)
        runs.append([b.read_particles(k) for k in (0, 1, extra)])
        calls = {k: v[1] for k, v in b.kernel_times().items()}
        b.close()
    for a, c in zip(*runs):
        for f in ("position", "velocity", "affine", "deformation"):
            assert np.array_equal(getattr(a, f), getattr(c, f)), f
    # the block table is cleared by a launch of its own where lists were made and lost unused
    if steps == 1:
        assert calls.get("k_bin_update", 0) == 0 and calls["k_topo_clear"] <= 1 + 48 // 16 + 1
    else:  # every second substep runs on lists
        assert calls["k_bin_update"] >= 40
