"""The one-pass compact form at the edges of its 512-slot tiles, over tiles of
several segments, and with arrays that are too small: exact round trips, and
no store past a cap."""
import ctypes

import numpy as np
import pytest

from pipeline_amd import OCP_OK, COMPACT_NODE_DTYPE, OcpError, clouds

pytestmark = pytest.mark.gpu
OCP_ERR_CAPACITY = 3


def _compact(ctx, nodes, node_cap, children, child_cap):
    kn, kc = ctypes.c_int64(-1), ctypes.c_int64(-1)
    rc = ctx.lib.ocp_compact_octree(ctx.h, nodes.ptr if nodes else None, node_cap,
                                    children.ptr if children else None, child_cap,
                                    ctypes.byref(kn), ctypes.byref(kc))
    return rc, kn.value, kc.value


@pytest.mark.parametrize("n", [1, 2, 900, 1050, 1100, 20_000, 400_000])
def test_round_trip_and_caps(ctx, n):
    d = ctx.upload(clouds.uniform(n, seed=n))
    ctx.build(d, n, 0.0, 1024.0)
    ref = ctx.fetch().nodes[0].view(np.uint8)
    rc, kn, kc = _compact(ctx, None, 0, None, 0)
    assert rc == OCP_OK and kn * 60 == ref.size
    assert kc == int((ctx.fetch().nodes[0]["children"] != 0).sum())
    guard = np.full(64, 7, np.uint8)
    nodes = ctx.upload(np.full(kn * 12 + 64, 7, np.uint8))
    children = ctx.upload(np.full(kc * 4 + 64, 7, np.uint8))
    assert _compact(ctx, nodes, kn, children, kc) == (OCP_OK, kn, kc)
    np.testing.assert_array_equal(nodes.to_host()[kn * 12:], guard)
    np.testing.assert_array_equal(children.to_host()[kc * 4:], guard)
    whole = children.to_host()
    cn = nodes.to_host()[:kn * 12].view(COMPACT_NODE_DTYPE)
    used = cn["child_set"][:, None] >> np.arange(8) & 1
    np.testing.assert_array_equal(cn["first_child"], np.concatenate([[0], used.sum(1).cumsum()[:-1]]))
    nodes.shape, nodes.dtype = (kn,), COMPACT_NODE_DTYPE
    children.shape, children.dtype = (kc,), np.dtype(np.int32)
    out = ctx.expand_octree(nodes, children, ctx.results().oct_start, 1)
    np.testing.assert_array_equal(out.to_host(kn * 60), ref)
    if kc > 1:  # too small: refused, with the sizes, and nothing past the cap
        children.copy_from(np.full(kc, 0x07070707, np.int32))
        assert _compact(ctx, nodes, kn, children, kc // 2) == (OCP_ERR_CAPACITY, kn, kc)
        assert (children.to_host()[kc // 2:] == 0x07070707).all()
        assert _compact(ctx, nodes, kn - 1, children, kc) == (OCP_ERR_CAPACITY, kn, kc)
    assert whole.size
    u, k = ctx.counts(1)  # the build's counts are still there
    assert int(k[0]) == kn
    for a in (d, nodes, children, out):
        a.free()


def test_many_small_segments(ctx):
    """Tiles that hold slots of many segments, each with its own box."""
    sizes = [1, 3, 40, 700, 2, 5, 300, 1, 1, 9000, 64] * 9
    pts = np.concatenate([clouds.clustered(s, seed=k) if s > 30 else clouds.uniform(s, seed=k)
                          for k, s in enumerate(sizes)])
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    rg = np.linspace(1024.0, 1500.0, len(sizes)).astype(np.float32)
    d = ctx.upload(pts)
    ctx.build_batched(d, offs, np.full(len(sizes), -3.0, np.float32), rg)
    r = ctx.results()
    ref = np.concatenate([v.view(np.uint8) for v in ctx.fetch(offs).nodes])
    nodes, children = ctx.compact_octree()
    out = ctx.expand_octree(nodes, children, r.oct_start, len(sizes), r.seg_min, r.seg_range)
    np.testing.assert_array_equal(out.to_host(ref.size), ref)
    for a in (d, nodes, children, out):
        a.free()


def test_wait_gives_up(ctx):
    n = 300_000
    d = ctx.upload(clouds.uniform(n, seed=1))
    ctx.build(d, n, 0.0, 1024.0)
    ctx.counts(1)
    try:
        ctx.set_wait_limit(0)
        with pytest.raises(OcpError, match="wait gave up"):
            ctx.compact_octree()
        ctx.set_wait_limit(-1)
        ctx.build(d, n, 0.0, 1024.0)
        nodes, children = ctx.compact_octree()
        nodes.free()
        children.free()
    finally:
        ctx.set_wait_limit(-1)
        d.free()
