"""The compact form of one pipeline slot while another builds: it has no wait
between workgroups, so it needs no order among the frames' waits."""
import numpy as np
import pytest

import oracle
from pipeline_amd import Pipeline, clouds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1050, 300_000])
def test_compact_waits_for_no_workgroup(n):
    pts = clouds.uniform(n, seed=n)
    ref = oracle.build_plain(pts)["nodes"].view(np.uint8)
    with Pipeline(2, max_points=n) as ppl:
        ctx = ppl.context(0)
        d = ctx.upload(pts)
        ppl.submit(0, d, n)
        ppl.wait(0)
        ctx.set_wait_limit(0)  # a wait would give up at once
        ppl.submit(1, d, n)
        nodes, children = ctx.compact_octree()
        ppl.wait(1)
        ctx.set_wait_limit(-1)
        out = ctx.expand_octree(nodes, children, ctx.results().oct_start, 1)
        np.testing.assert_array_equal(out.to_host(ref.size), ref)
        np.testing.assert_array_equal(ppl.context(1).fetch().nodes[0].view(np.uint8), ref)
        for a in (d, nodes, children, out):
            a.free()
