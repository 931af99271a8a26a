"""The default tile table stands for the library's own choice of the path:
after a save and restore, and where the autotuner finds nothing faster."""
import numpy as np
import pytest

import oracle
import pipeline_amd
from pipeline_amd import clouds
from test_gpu_pipeline import _check_segment

pytestmark = pytest.mark.gpu


def _sort_kernels(ctx, d, n):
    ctx.set_stage_timing(True)
    ctx.build(d, n, 0.0, 1024.0)
    ctx.set_stage_timing(False)
    return set(ctx.kernel_ms())


def test_restored_table_keeps_the_choice():
    n = 100_000
    pts = clouds.uniform(n, seed=2)
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(pts)
        own = _sort_kernels(ctx, d, n)
        assert "msd_scatter" in own
        base = ctx.get_tune()
        ctx.set_tune(**base)
        assert _sort_kernels(ctx, d, n) == own
        ctx.set_tune(scan_ipt=8)  # a table: its 8-bit passes stand
        assert "msd_scatter" not in _sort_kernels(ctx, d, n)
        ctx.set_tune(**base)
        assert _sort_kernels(ctx, d, n) == own
        _check_segment(ctx.fetch(), 0, oracle.build_plain(pts))
    for size in (n, 10_000_000):
        assert pipeline_amd.workspace_size(size, tune=base) == pipeline_amd.workspace_size(size)


def test_autotune_keeps_the_choice_of_small_clouds(tmp_path):
    """One kernel before the octree takes less than half the stages' time, which
    is all that a table can give."""
    pts = clouds.uniform(4096, seed=4)
    with pipeline_amd.Context(0) as ctx:
        base = ctx.get_tune()
        d = ctx.upload(pts)
        cache = str(tmp_path / "tune.txt")
        assert ctx.autotune(d, reps=5, cache=cache) == base and ctx.get_tune() == base
        big = clouds.uniform(100_000, seed=5)
        db = ctx.upload(big)
        assert "msd_scatter" in _sort_kernels(ctx, db, 100_000)
        assert ctx.autotune(d, reps=5, cache=cache) == base and ctx.tune_from_cache
        assert "msd_scatter" in _sort_kernels(ctx, db, 100_000)
        ctx.build(d, 4096, 0.0, 1024.0)
        _check_segment(ctx.fetch(), 0, oracle.build_plain(pts))
