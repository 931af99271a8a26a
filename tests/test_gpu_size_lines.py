"""Builds on both sides of every line of size that a new context's choices have
above the smallest, and the crowded keys' switch of the sort in batches, from
graphs and after its run of builds, against the oracle."""
import numpy as np
import pytest

import oracle
import pipeline_amd
from test_gpu_pipeline import _check_segment
from test_gpu_tree_tiles import _cells

pytestmark = pytest.mark.gpu


# 2800 and 6000 keys a digit; nodes past the caches; the offsets kernel
@pytest.mark.parametrize("n", [2_867_200, 2_867_201, (1 << 22) - 1, 1 << 22, 6_144_000, 6_144_001,
                               (1 << 23) - 1, 1 << 23])
def test_one_cloud(n):
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 1 << 30, n)
    keys[: n // 8] = keys[n // 8: 2 * (n // 8)]  # some twice
    pts = _cells(keys)
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(pts)
        ctx.build(d, n, 0.0, 1024.0)
        _check_segment(ctx.fetch(), 0, oracle.build_plain(pts))


@pytest.mark.parametrize("graph", [False, True])
def test_crowded_batch_changes_its_sort(graph):
    rng = np.random.default_rng(4)
    sizes = [40_000, 20_000, 3000, 50_000]
    pts = [_cells((700 << 20) + rng.integers(0, 1 << 19, s)) for s in sizes]
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    exp = [oracle.build_plain(p) for p in pts]
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(np.concatenate(pts))
        ctx.set_graph_mode(graph)
        for _ in range(4):  # (the counts are read with the outputs)
            ctx.build_batched(d, offs, [0.0] * 4, [1024.0] * 4)
            out = ctx.fetch(offs)
            for k in range(4):
                _check_segment(out, k, exp[k])


def test_switch_ends():
    """256 builds after the counts have told, then the first sort again."""
    rng = np.random.default_rng(6)
    pts = _cells((700 << 20) + rng.integers(0, 1 << 19, 20_000))
    exp = oracle.build_plain(pts)
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(pts)

        def msd():
            ctx.set_stage_timing(True)
            ctx.build(d, pts.shape[0], 0.0, 1024.0)
            ctx.set_stage_timing(False)
            _check_segment(ctx.fetch(), 0, exp)
            return "msd_scatter" in ctx.kernel_ms()
        assert msd()
        assert not msd()
        for _ in range(255):
            ctx.build(d, pts.shape[0], 0.0, 1024.0)
        assert msd()
        assert not msd()
