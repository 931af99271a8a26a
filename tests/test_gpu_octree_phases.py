"""The make and link entries one by one, at the edges of the octree kernel's
tiles of 512 nodes, with chains and walks that cross them, and with more slots
than the chains use, against the oracle's sequential phases."""
import numpy as np
import pytest

import oracle
from pipeline_amd import OCT_NODE_DTYPE
from test_gpu_stages import _unique_codes

pytestmark = pytest.mark.gpu

MN, RG = -40.0, 256.0


def _phases(codes, tree, e, p, k):
    """Nodes after the root setup and make, and after link."""
    ptr = lambda a: a.ctypes.data
    nodes = np.zeros(k, OCT_NODE_DTYPE)
    lib, m = oracle.lib(), e.size
    lib.orc_root_init(ptr(nodes), ptr(codes), ptr(tree["prefix_n"]), m, MN, RG)
    lib.orc_make_oct_nodes(ptr(nodes), ptr(p), ptr(e), ptr(codes), ptr(tree["prefix_n"]),
                           ptr(tree["parent"]), MN, RG, m, k, 1)
    made = nodes.copy()
    lib.orc_link_leaf_nodes(ptr(nodes), ptr(p), ptr(e), ptr(codes), ptr(tree["has_leaf_left"]),
                            ptr(tree["has_leaf_right"]), ptr(tree["prefix_n"]),
                            ptr(tree["parent"]), ptr(tree["left_child"]), m, k, 1)
    return made, nodes


def _codes(u, kind):
    pair = np.arange(u // 2) * ((1 << 30) // u)
    return np.unique({
        "consecutive": np.arange(u),
        "sparse": np.arange(u) * ((1 << 30) // u),
        "pairs": np.concatenate([pair, pair + 1]),
        "corner": np.concatenate([np.arange(max(u - 25, 1)), 1 << np.arange(10, 30)]),
        "uniform": _unique_codes(u, u) if u > 100 else np.arange(u) * 12345,
        "clustered": _unique_codes(u, u, "clustered") if u > 100 else np.arange(u) * 54321,
    }[kind]).astype(np.uint32)


@pytest.mark.parametrize("kind", ["consecutive", "sparse", "pairs", "corner", "uniform",
                                  "clustered"])
@pytest.mark.parametrize("u", [2, 3, 512, 513, 514, 1025, 1026, 9000])
def test_make_then_link(ctx, u, kind):
    codes = _codes(u, kind)
    tree = oracle.build_radix_tree(codes)
    e = oracle.edge_count(tree["prefix_n"], tree["parent"])
    p = oracle.partial_sum(e)
    used = int(oracle.octree(codes, tree, e, p)[1])
    dev = {k: ctx.upload(v) for k, v in tree.items()}
    de, dp, dc = ctx.upload(e), ctx.upload(p), ctx.upload(codes)
    m = e.size
    for k in (used, used + 700):
        made, linked = _phases(codes, tree, e, p, k)
        nodes = ctx.upload(np.full(k * 15, 0x5A5A5A5A, np.int32))
        ctx.k_InitOctNodes(nodes, k, dc, dev["prefix_n"], m, MN, RG)
        ctx.k_MakeOctNodes(nodes, dp, de, dc, dev["prefix_n"], dev["parent"], MN, RG, m, k)
        np.testing.assert_array_equal(nodes.to_host().view(np.uint8), made.view(np.uint8))
        ctx.k_LinkLeafNodes(nodes, dp, de, dc, dev["has_leaf_left"], dev["has_leaf_right"],
                            dev["prefix_n"], dev["parent"], dev["left_child"], m, k)
        np.testing.assert_array_equal(nodes.to_host().view(np.uint8), linked.view(np.uint8))
        nodes.free()
    for a in (*dev.values(), de, dp, dc):
        a.free()
