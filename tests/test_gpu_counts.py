"""Counts after a build come from host memory that the build itself writes:
as many segments as it holds and one more, and per-stage work between a build
and its counts, against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _expect(pts, offs):
    q = pts[:, :3].astype(np.int64)
    ids = (q[:, 0] << 20) | (q[:, 1] << 10) | q[:, 2]
    return np.array([np.unique(ids[a:b]).size for a, b in zip(offs[:-1], offs[1:])], np.int32)


@pytest.mark.parametrize("n_seg", [1, 2, 4096, 4097])
def test_counts_per_segment(ctx, n_seg):
    rng = np.random.default_rng(n_seg)
    offs = np.concatenate([[0], np.cumsum(rng.integers(1, 6, n_seg))]).astype(np.int32)
    pts = np.zeros((offs[-1], 4), np.float32)
    pts[:, :3] = rng.integers(0, 3, (offs[-1], 3)) * 500
    want = _expect(pts, offs)
    d, keys, alt = ctx.upload(pts), ctx.zeros(1000, np.uint32), ctx.zeros(1000, np.uint32)
    try:
        for _ in range(2):
            ctx.build_batched(d, offs, [0.0] * n_seg, [1024.0] * n_seg)
            u, k = ctx.counts(n_seg)
            np.testing.assert_array_equal(u, want)
            assert (k >= 1).all()
            ctx.k_SortKeys(keys, alt, 1000)  # the mail is no longer the last word
            u2, k2 = ctx.counts(n_seg)
            np.testing.assert_array_equal(u2, u)
            np.testing.assert_array_equal(k2, k)
    finally:
        for a in (d, keys, alt):
            a.free()
