"""A compact call that is refused stores nothing, whichever of its caps is too
small, and where slots have no exact form."""
import numpy as np
import pytest

from pipeline_amd import OCP_OK, Pipeline, clouds
from test_gpu_compact_edges import OCP_ERR_CAPACITY, _compact

pytestmark = pytest.mark.gpu
OCP_ERR_STATE = 4


@pytest.mark.parametrize("n", [30, 1050, 400_000])
@pytest.mark.parametrize("slot", [False, True])
def test_small_arrays(ctx, n, slot):
    with Pipeline(1, max_points=n) as ppl:
        c = ppl.context(0) if slot else ctx
        d = c.upload(clouds.uniform(n, seed=n))
        c.build(d, n, 0.0, 1024.0)
        rc, kn, kc = _compact(c, None, 0, None, 0)
        assert rc == OCP_OK
        nodes = c.upload(np.full(kn * 12, 7, np.uint8))
        children = c.upload(np.full(kc * 4, 7, np.uint8))
        for node_cap, child_cap in ((kn, kc - 1), (kn, 0), (kn - 1, kc), (kn - 1, 10 * kc)):
            assert _compact(c, nodes, node_cap, children, child_cap) == (OCP_ERR_CAPACITY, kn, kc)
            assert (nodes.to_host() == 7).all() and (children.to_host() == 7).all()
        assert _compact(c, nodes, kn, children, kc) == (OCP_OK, kn, kc)
        exact = nodes.to_host(), children.to_host()
        roomy = c.upload(np.full((kn + n + 32) * 4, 7, np.uint8))  # the one pass
        assert _compact(c, nodes, kn, roomy, kn + n + 32) == (OCP_OK, kn, kc)
        np.testing.assert_array_equal(nodes.to_host(), exact[0])
        np.testing.assert_array_equal(roomy.to_host()[:kc * 4], exact[1])
        assert (roomy.to_host()[kc * 4:] == 7).all()
        for a in (d, nodes, children, roomy):
            a.free()


@pytest.mark.parametrize("auto", [False, True])
def test_box_without_exact_forms(ctx, auto):
    """Far from the origin corners round to fewer values than the grid has."""
    n = 100_000
    pts = clouds.uniform(n, seed=3)
    pts[:, :3] = pts[:, :3] * np.float32(7.3 / 1024.0) + np.float32(1.0e6)
    d = ctx.upload(pts)
    if auto:
        ctx.build_autobox(d, n)
    else:
        ctx.build(d, n, 1.0e6, 7.3)
    k = int(ctx.counts(1)[1][0])
    nodes = ctx.upload(np.full(k * 12, 7, np.uint8))
    children = ctx.upload(np.full((k + n + 32) * 4, 7, np.uint8))
    rc, kn, _ = _compact(ctx, nodes, k, children, k + n + 32)
    assert (rc, kn) == (OCP_ERR_STATE, k)
    assert (nodes.to_host() == 7).all() and (children.to_host() == 7).all()
    for a in (d, nodes, children):
        a.free()
