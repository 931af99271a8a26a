"""The sort form that a build takes by itself (windows of the top digit's
scatter sorted in LDS, a second level for digits too large for it): the rule's
line, and key sets that reach each way a digit is sorted. Every stage output
against the oracle, eager and from a graph."""
import numpy as np
import pytest

import oracle
import pipeline_amd
from test_gpu_pipeline import _check_segment
from test_gpu_tree_tiles import _cells

pytestmark = pytest.mark.gpu


def _keys(kind, rng):
    if kind == "equal":                 # one key: one run above 65,536
        return np.full(100_000, 123_456_789)
    if kind == "two runs":              # two long runs of one digit, and a short one
        return np.concatenate([np.full(70_000, 5 << 20), (5 << 20) + (3 << 10) + rng.integers(0, 7, 90_000),
                               (5 << 20) + (9 << 10) + rng.integers(0, 1024, 20_000)])
    if kind == "block and a stray":     # a dense block in one corner of the box
        return np.append(rng.integers(0, 3000, 200_000), (1 << 30) - 1)
    if kind == "one digit":             # second-level digits of a few keys each
        return (700 << 20) + rng.integers(0, 1 << 20, 150_000)
    if kind == "few digits":            # digits at and about the LDS capacity
        sizes = [4095, 4096, 4097, 1, 12287, 12288, 12289, 8192, 8193, 20_000]
        return np.concatenate([(k * 37 << 20) + rng.integers(0, 1 << 20, s)
                               for k, s in enumerate(sizes)])
    if kind == "prefix sizes":          # one-prefix runs about a window and the LDS capacity
        sizes = [8191, 8192, 8193, 12288, 12289, 65_536, 65_537, 40, 4000]
        return np.concatenate([(3 << 20) + (k * 11 << 10) + rng.integers(0, 1024, s)
                               for k, s in enumerate(sizes)])
    return rng.integers(0, 1 << 30, 300_000)


KINDS = ["equal", "two runs", "block and a stray", "one digit", "few digits", "prefix sizes",
         "uniform"]


@pytest.mark.parametrize("kind", KINDS)
def test_key_sets(kind):
    rng = np.random.default_rng(len(kind))
    pts = _cells(rng.permutation(_keys(kind, rng)))
    exp = oracle.build_plain(pts)
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(pts)
        for graph in (False, True):
            ctx.set_graph_mode(graph)
            for _ in range(3):
                ctx.build(d, pts.shape[0], 0.0, 1024.0)
                _check_segment(ctx.fetch(), 0, exp)


def test_large_cloud_with_every_kind():
    """Above 2800 keys a digit the windows and the capacity are the larger
    ones."""
    rng = np.random.default_rng(11)
    keys = np.concatenate([_keys(k, rng) for k in KINDS] + [rng.integers(0, 1 << 30, 2_500_000)])
    pts = _cells(rng.permutation(keys))
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(pts)
        ctx.build(d, pts.shape[0], 0.0, 1024.0)
        _check_segment(ctx.fetch(), 0, oracle.build_plain(pts))


@pytest.mark.parametrize("n", [16_383, 16_384, 16_385, 65_537])
def test_rule_line(n):
    pts = _cells(np.random.default_rng(n).integers(0, 1 << 30, n))
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(pts)
        ctx.build(d, n, 0.0, 1024.0)
        _check_segment(ctx.fetch(), 0, oracle.build_plain(pts))


def test_batch_of_every_kind():
    rng = np.random.default_rng(5)
    sets = [_keys(k, rng) for k in KINDS] + [np.zeros(0, np.int64), np.array([7])]
    pts = [_cells(rng.permutation(s)) for s in sets]
    offs = np.concatenate([[0], np.cumsum([p.shape[0] for p in pts])]).astype(np.int32)
    with pipeline_amd.Context(0) as ctx:
        d = ctx.upload(np.concatenate(pts))
        ctx.build_batched(d, offs, [0.0] * len(pts), [1024.0] * len(pts))
        out = ctx.fetch(offs)
        for k, p in enumerate(pts):
            if p.shape[0]:
                _check_segment(out, k, oracle.build_plain(p))


@pytest.mark.parametrize("n", [20_000, 300_000, 2_999_999, 3_000_000])
def test_builds_after_crowded_keys(n):
    """Once the counts of a build have told that its keys crowd, the next of
    about its size take LSD passes; 3M points is the line between their widths."""
    rng = np.random.default_rng(n)
    sets = [_cells((700 << 20) + rng.integers(0, 1 << 20, m)) for m in (n, n, n - n // 3)]
    with pipeline_amd.Context(0) as ctx:
        for pts in sets:
            d = ctx.upload(pts)
            ctx.build(d, pts.shape[0], 0.0, 1024.0)
            _check_segment(ctx.fetch(), 0, oracle.build_plain(pts))
