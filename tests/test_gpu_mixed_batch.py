"""Batches of one long cloud and many short ones: the windows of the sort go by
each cloud's own length."""
import numpy as np
import pytest

import oracle
import pipeline_amd
from pipeline_amd import clouds
from test_gpu_pipeline import _check_segment

pytestmark = pytest.mark.gpu


def _batch(sizes):
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    pts = np.concatenate([clouds.clustered(s, seed=k) if k % 3 == 1 and s > 30
                          else clouds.uniform(s, seed=k) for k, s in enumerate(sizes) if s])
    return offs, pts


def test_outputs():
    """Both sides of the line at 6,144,000 points, and clouds about a window."""
    sizes = [5, 6_144_001, 0, 4095, 4096, 4097, 300_000, 1, 20_000]
    offs, pts = _batch(sizes)
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(pts)
        ctx.build_batched(d, offs, [0.0] * len(sizes), [1024.0] * len(sizes))
        out = ctx.fetch(offs)
        for k, s in enumerate(sizes):
            if s:
                _check_segment(out, k, oracle.build_plain(pts[offs[k]:offs[k + 1]]))


def test_short_clouds_cost_little():
    """2000 clouds of 100 points beside one of 6.2M: with a workgroup a digit for
    each of them the batch took 25 times the long cloud's build."""
    n = 6_200_000
    sizes = [n] + [100] * 2000
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(clouds.uniform(int(offs[-1]), seed=1))
        alone = ctx.time_builds(d, n=n, warmup=3, steps=10)
        box = [0.0] * len(sizes), [1024.0] * len(sizes)
        batch = ctx.time_builds(d, seg_offsets=offs, seg_min=box[0], seg_range=box[1], warmup=3,
                                steps=10)
        assert batch < 4 * alone, (batch, alone)


def test_small_build_after_a_large_one():
    """What a context has room for must not cost the builds that need little."""
    n, large = 20_000, 100_000_000
    with pipeline_amd.Context(0) as ctx:
        d = ctx.empty((large, 4), np.float32)
        ctx.k_InitRandomVec4(d, large, 0.0, 1024.0, 1)

        def best():
            return min(ctx.time_builds(d, n=n, warmup=10, steps=50) for _ in range(5))
        before = best()
        ctx.build(d, large, 0.0, 1024.0)
        ctx.synchronize()
        after = best()
        assert after < 1.25 * before, (before, after)
        ctx.build(d, n, 0.0, 1024.0)
        _check_segment(ctx.fetch(), 0, oracle.build_plain(d.to_host(n * 4).reshape(n, 4)))
