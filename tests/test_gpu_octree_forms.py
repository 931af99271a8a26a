"""The make and link entries on arrays of other forms than a build's, against
the oracle's sequential phases."""
import numpy as np
import pytest

import oracle
from test_gpu_octree_phases import MN, RG, _codes, _phases

pytestmark = pytest.mark.gpu


def _check(ctx, codes, tree, e, p, k):
    """Both entries on k nodes against the oracle."""
    made, linked = _phases(codes, tree, e, p, k)
    dev = {f: ctx.upload(v) for f, v in tree.items()}
    de, dp, dc = ctx.upload(e), ctx.upload(p), ctx.upload(codes)
    nodes = ctx.upload(np.full(k * 15, 0x5A5A5A5A, np.int32))
    m = e.size
    try:
        ctx.k_InitOctNodes(nodes, k, dc, dev["prefix_n"], m, MN, RG)
        ctx.k_MakeOctNodes(nodes, dp, de, dc, dev["prefix_n"], dev["parent"], MN, RG, m, k)
        np.testing.assert_array_equal(nodes.to_host().view(np.uint8), made.view(np.uint8))
        ctx.k_LinkLeafNodes(nodes, dp, de, dc, dev["has_leaf_left"], dev["has_leaf_right"],
                            dev["prefix_n"], dev["parent"], dev["left_child"], m, k)
        np.testing.assert_array_equal(nodes.to_host().view(np.uint8), linked.view(np.uint8))
    finally:
        for a in (*dev.values(), de, dp, dc, nodes):
            a.free()


def _offsets(form, e, rng):
    """First slots of every chain, slot 0 the root's."""
    if form == "inclusive":
        return oracle.partial_sum(e)
    if form == "shifted":  # overlapping as the inclusive scan's, 7 slots on
        p = oracle.partial_sum(e) + 7
    elif form == "exclusive":  # no two chains share a slot
        p = np.cumsum(e) - e + 1
    elif form == "gaps":
        room = e + rng.integers(0, 4, e.size)
        p = np.cumsum(room) - room + 1
    else:  # "reversed": the last chain first
        p = 1 + int(e.sum()) - np.cumsum(e)
    p[0] = 0
    return p.astype(np.int32)


@pytest.mark.parametrize("form", ["inclusive", "shifted", "exclusive", "gaps", "reversed"])
@pytest.mark.parametrize("u", [3, 513, 1030, 20000])
def test_offsets_of_any_form(ctx, form, u):
    rng = np.random.default_rng(u)
    for kind in ("uniform", "clustered"):
        codes = _codes(u, kind)
        tree = oracle.build_radix_tree(codes)
        e = oracle.edge_count(tree["prefix_n"], tree["parent"])
        p = _offsets(form, e, rng)
        used = max(1, int((p + e).max()))
        for k in (used, used + 90, max(1, used - used // 5)):
            _check(ctx, codes, tree, e, p, k)


def _repeated(kind, u):
    """Sorted codes with repeats."""
    base = _codes(u, "uniform")
    mid = base[base.size // 2]
    return {"one code": lambda: np.full(u, mid), "one pair": lambda: np.append(base, mid),
            "twice": lambda: np.repeat(base[:u // 2 + 1], 2),
            "run": lambda: np.append(base, np.full(700, mid))}[kind]()


@pytest.mark.parametrize("kind", ["one code", "one pair", "twice", "run"])
@pytest.mark.parametrize("u", [513, 1400, 5400])
def test_repeated_codes(ctx, kind, u):
    """The tree over codes that repeat, which its entry takes: chains by the
    inclusive scan, children that are no node, nodes that name each other."""
    codes = np.sort(_repeated(kind, u)).astype(np.uint32)
    tree = oracle.build_radix_tree(codes)
    e = oracle.edge_count(tree["prefix_n"], tree["parent"])
    p = oracle.partial_sum(e)
    assert e.min() >= 0 and p[0] == 0
    _check(ctx, codes, tree, e, p, max(1, int((p + e).max())))


@pytest.mark.parametrize("bits", ["30", "30 or not", "31"])
@pytest.mark.parametrize("u", [3, 513, 3000])
def test_codes_of_more_than_30_bits(ctx, bits, u):
    base = _codes(u, "uniform").astype(np.uint64)
    some = np.random.default_rng(u).integers(0, 2, base.size).astype(np.uint64)
    top = {"30": 1 << 30, "30 or not": some << np.uint64(30), "31": 1 << 31}[bits]
    codes = np.sort(base + top).astype(np.uint32)
    tree = oracle.build_radix_tree(codes)
    e = oracle.edge_count(tree["prefix_n"], tree["parent"])
    p = oracle.partial_sum(e)
    _check(ctx, codes, tree, e, p, max(1, int((p + e).max())))
