"""The kernel names of a build stay what they were when other work follows it."""
import numpy as np
import pytest

import pipeline_amd
from test_gpu_tree_tiles import _cells

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("crowded", [False, True])
def test_names_after_other_work(crowded):
    rng = np.random.default_rng(2)
    keys = rng.integers(0, 1 << (20 if crowded else 30), 100_000)
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(_cells(keys))
        ctx.set_stage_timing(True)
        ctx.build(d, keys.size, 0.0, 1024.0)
        names = set(ctx.kernel_ms())
        assert ("msd_lsd_fallback" if crowded else "msd_lsd_skipped") in names
        ctx.compact_octree()
        assert set(ctx.kernel_ms()) == names
        k, alt = ctx.zeros(40_000, np.uint32), ctx.zeros(40_000, np.uint32)
        ctx.k_SortKeys(k, alt, 40_000)
        assert set(ctx.kernel_ms()) == names
