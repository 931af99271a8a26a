"""Clouds whose stages 1 to 6 run in one workgroup (at most 8192 points per
cloud) and the kernels of those stages (the same builds with stage timing on):
all stage outputs against the oracle, either side of the kernel's two
capacities."""
import numpy as np
import pytest

import oracle
from pipeline_amd import clouds
from test_gpu_pipeline import _check_segment
from test_gpu_tree_tiles import _cells

pytestmark = pytest.mark.gpu


def _both_ways(ctx, pts, exp):
    d = ctx.upload(pts)
    try:
        for timing in (False, True):
            ctx.set_stage_timing(timing)
            ctx.build(d, pts.shape[0], 0.0, 1024.0)
            u, k = ctx.counts(1)
            assert (int(u[0]), int(k[0])) == (exp["n_unique"], exp["n_oct"])
            _check_segment(ctx.fetch(), 0, exp)
    finally:
        ctx.set_stage_timing(False)
        d.free()


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 257, 1023, 1025, 4095, 4096, 4097, 5121, 8191,
                               8192, 8193])
def test_sizes(ctx, n):
    for pts in (clouds.uniform(n, seed=n, float4=False), clouds.clustered(n, seed=n),
                np.tile(np.float32([[700.5, 2.5, 3.5, 0.0]]), (n, 1))):
        _both_ways(ctx, pts, oracle.build_plain(pts))


@pytest.mark.parametrize("n", [2, 3, 63, 1023, 4095, 4096, 4097, 9999, 16383, 16384, 16385,
                               (1 << 20) - 1, 1 << 20])
def test_key_sort_sizes(ctx, n):
    """The sort entry around what one workgroup takes and where its first pass
    changes form: spread, crowded, equal and full 32-bit keys."""
    rng = np.random.default_rng(n)
    for keys in (rng.integers(0, 1 << 30, n), rng.integers(0, 1 << 32, n),
                 rng.integers(0, 50, n) + (rng.integers(0, 3, n) << 28), np.full(n, 0xffffffff)):
        keys = keys.astype(np.uint32)
        a, b = ctx.upload(keys), ctx.empty(n, np.uint32)
        ctx.k_SortKeys(a, b, n)
        np.testing.assert_array_equal(a.to_host(), np.sort(keys))
        a.free()
        b.free()


@pytest.mark.parametrize("u", [511, 2049, 4096, 8192])
def test_code_patterns(ctx, u):
    """Consecutive codes, powers of two apart, far pairs, and a crowd of codes
    in a few places (the sort's radix passes)."""
    pair = np.arange(u // 2) * ((1 << 30) // u)
    for keys in (np.arange(u), (1 << 30) - 1 - np.arange(u), np.arange(u) * ((1 << 30) // u),
                 np.concatenate([pair, pair + 1]),
                 np.concatenate([np.arange(u - 25) // 2, 1 << np.arange(5, 30)])):
        pts = _cells(np.random.default_rng(u).permutation(keys))
        _both_ways(ctx, pts, oracle.build_plain(pts))


@pytest.mark.parametrize("hi", [4096, 8192, 8193])
def test_batches_and_boxes(ctx, hi):
    """Clouds of 0 to hi points with boxes of their own, given and found, and
    in a replayed graph with new points in the same buffer."""
    rng = np.random.default_rng(hi)
    sizes = np.concatenate([[0, 1, hi, 2, 0], rng.integers(1, hi, 20), [0]])
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    d = None
    try:
        for rep in range(3):
            pts = clouds.uniform(int(offs[-1]), seed=rep)
            pts[:, :3] = pts[:, :3] * np.float32(0.3) - np.float32(50 + rep)
            smin = np.full(sizes.size, -50.0 - rep, np.float32)
            srg = np.full(sizes.size, 310.0, np.float32)
            if d is None:
                d = ctx.upload(pts)
            else:
                d.copy_from(pts)
            ctx.set_graph_mode(rep > 0)
            for given in (True, False):
                if given:
                    ctx.build_batched(d, offs, smin, srg)
                else:
                    ctx.build_batched(d, offs)
                out = ctx.fetch(offs)
                for s in range(sizes.size):
                    p = pts[offs[s]:offs[s + 1]]
                    if p.shape[0] == 0:
                        assert int(out.n_unique[s]) == 0 and int(out.n_oct[s]) == 0
                        continue
                    mn, rg = (smin[s], srg[s]) if given else clouds.cube_box(p)
                    _check_segment(out, s, oracle.build_plain(p, float(mn), float(rg)))
        ctx.set_graph_mode(False)
        one = int(sizes[2])
        ctx.build_autobox(d, one)
        mn, rg = clouds.cube_box(pts[:one])
        _check_segment(ctx.fetch(), 0, oracle.build_plain(pts[:one], float(mn), float(rg)))
    finally:
        ctx.set_graph_mode(False)
        if d is not None:
            d.free()
