"""The fused build's radix tree and octree at the edges of their tiles (tree:
512 nodes below 2^21 points, 2048 from there; octree: 512): segment ends at,
before and after a tile end and a window end, codes whose nodes reach past the
window, and tiles with more octree slots than the kernel keeps at once, all
stage outputs against the oracle."""
import numpy as np
import pytest

import oracle
from pipeline_amd import clouds
from test_gpu_pipeline import _check_segment, _plain

pytestmark = pytest.mark.gpu


def _cells(keys):
    """Points whose Morton keys are the given ones (box [0, 1024))."""
    k = np.asarray(keys, np.uint64)
    pts = np.zeros((k.size, 4), np.float32)
    for axis in range(3):
        q = np.zeros(k.size, np.uint64)
        for b in range(10):
            q |= ((k >> np.uint64(3 * b + axis)) & np.uint64(1)) << np.uint64(b)
        pts[:, axis] = q.astype(np.float32) + np.float32(0.5)
    return pts


@pytest.mark.parametrize("u", [2, 3, 511, 512, 513, 514, 1023, 1024, 1025, 1026, 1537, 2049])
def test_consecutive_and_sparse_codes(ctx, u):
    """Runs of u codes: consecutive ones (every node a power of two wide) and
    powers of two apart (a chain: every node reaches one end)."""
    for keys in (np.arange(u), np.arange(u) * ((1 << 30) // u),
                 np.unique(np.concatenate([np.arange(max(u - 25, 1)), 1 << np.arange(10, 30)]))):
        pts = _cells(keys)
        _check_segment(_plain(ctx, pts), 0, oracle.build_plain(pts))


@pytest.mark.parametrize("n", [(1 << 21) - 1, 1 << 21, (1 << 21) + 2049])
def test_tile_rule(ctx, n):
    """Either side of the rule's line, with a dense corner and a sparse rest:
    nodes that reach thousands of keys to both sides."""
    rng = np.random.default_rng(n)
    keys = np.concatenate([np.arange(n // 2) + (1 << 29) - n // 4,
                           rng.integers(0, 1 << 30, n - n // 2)])
    pts = _cells(rng.permutation(keys))
    _check_segment(_plain(ctx, pts), 0, oracle.build_plain(pts))


@pytest.mark.parametrize("pairs,gap", [(40, 1 << 24), (700, 1 << 20), (5000, 1 << 17)])
def test_long_chains(ctx, pairs, gap):
    """Sibling pairs far apart: chains of up to nine slots, so a tile of 512
    nodes has several times the 320 slots of a round, and chains that start in
    one tile and cover slots of the next."""
    base = np.arange(pairs) * gap
    for extra in ([], [1 << 29], [(1 << 30) - 1]):
        keys = np.unique(np.concatenate([base, base + 1, np.asarray(extra, np.int64)]))
        pts = _cells(keys[keys < (1 << 30)])
        _check_segment(_plain(ctx, pts), 0, oracle.build_plain(pts))


def test_batched_odd_starts(ctx):
    """Segments that start at odd offsets (unaligned wide stores)."""
    sizes = [1, 2, 515, 1, 1029, 7, 2047, 3]
    pts = np.concatenate([clouds.uniform(s, seed=k) for k, s in enumerate(sizes)])
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    d = ctx.upload(pts)
    ctx.build_batched(d, offs, [0.0] * len(sizes), [1024.0] * len(sizes))
    out = ctx.fetch(offs)
    d.free()
    for s in range(len(sizes)):
        _check_segment(out, s, oracle.build_plain(pts[offs[s]:offs[s + 1]]))
