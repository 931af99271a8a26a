"""Performance cases of the octree pipeline: what its users have it do.

A case is a dict; ``prepare`` makes what a program holds before the call (a
context, its input in device memory, kept output buffers), ``run`` is one
pass through the public entry points, ``work`` the bytes it cannot do
without. The kinds of call:

frame    one cloud built whole and its counts read, as a program does per
         sensor frame before it uses the tree; plain, with the box reduced on
         the device, with the key->point permutation, replayed from a graph,
         with the default tile table or with one that was tuned earlier
batch    many uneven clouds in one segmented build, each with its own box
stages   the seven per-stage entries called one after the other with the
         caller's own buffers, as a caller of the reference's stage functions
stream   frames through the two-slot pipeline
sort     k_SortKeys (or k_SortPairs) on Morton keys
learned  sort_learned on Morton keys with a model trained on an earlier frame
compact  the last build's octree into the 12-byte node format
expand   the 12-byte node format back into 60-byte nodes

The calls that return before their work has ended are followed by the
context's synchronize, which reports their errors and without which another
stream may not read their results. Outputs are device buffers of the context
(or of the caller), whole. All of them are integers or node records, compared
as their words, so there is no 64-bit value to hold them against: ``exact``
is None throughout.
"""
from __future__ import annotations

import ctypes
import math

import torch

import pipeline_amd
from pipeline_amd import Context, Pipeline

MIN, RANGE = 0.0, 1024.0
LIMIT = 1023.99993896484375  # the largest float below 1024
NODE_BYTES = 60

# A tile table tuned for large uniform clouds (what the autotuner of the
# benchmark settles on at 10M points).
TUNED = {"sort_bits": 10, "sort_msd": 1, "sort10_kpt": 16, "morton_ppt": 16,
         "morton_grid": 512, "scan_ipt": 8}


# ---------------------------------------------------------------- cases
def listed():
    return [
        # The smallest cloud of the batch workload as a frame of its own:
        # launches and round trips to the host are all of it.
        _frame("frame_4k", n=4096),
        # The benchmark's CPU-path cloud (307,200 points, one depth image).
        _frame("frame_307k", n=307200),
        # An ordinary lidar-like frame whose owner wants to know which point
        # is behind each key and does not know its box: odd size, packed xyz.
        _frame("frame_1m_perm", n=1000003, cloud="clustered", width=3, permutation=True,
               autobox=True),
        # The headline workload as the benchmark runs it: tuned, from a graph.
        _frame("frame_10m_tuned", n=10000000, graph=True, tuned=True),
        # The clustered scene of 2^24 points, with what a new context does.
        _frame("scene_16m", n=1 << 24, cloud="clustered", width=3),
        # A server's batch: clouds of 4,096 to 512K points, mixed kinds.
        {"name": "batch_64", "kind": "batch", "clouds": 64, "lo": 4096, "hi": 524288, "width": 4,
         "graph": True, "boxes": True},
        # A caller of the per-stage functions, with buffers of its own.
        {"name": "stages_2m", "kind": "stages", "n": 2000003, "cloud": "uniform", "width": 4},
        # Frames arriving faster than they are built.
        {"name": "stream_1m", "kind": "stream", "n": 1 << 20, "cloud": "uniform", "frames": 8},
        # The sort alone, keys of the clustered scene.
        {"name": "sort_16m", "kind": "sort", "n": 1 << 24, "cloud": "clustered", "pairs": False},
        # The learned sort on the next frame of a scene.
        {"name": "learned_32m", "kind": "learned", "n": 1 << 25, "cloud": "clustered"},
        # Storing an octree, and reading one back.
        {"name": "compact_2m", "kind": "compact", "n": 1 << 21, "cloud": "uniform"},
        {"name": "expand_2m", "kind": "expand", "n": 1 << 21, "cloud": "uniform"},
    ]


def _frame(name, n, cloud="uniform", width=4, permutation=False, autobox=False, graph=False,
           tuned=False):
    case = {"kind": "frame", "n": n, "cloud": cloud, "width": width,
            "permutation": permutation, "autobox": autobox, "graph": graph, "tuned": tuned}
    return {"name": name, **case} if name else case


def _log_size(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "batch", "stages", "stream", "sort",
                       "learned", "compact", "expand"])
    cloud = rng.choice(["uniform", "clustered"])
    width = rng.choice([3, 4])
    if kind == "frame":
        n = _log_size(rng, 700, 12000000)
        return _frame(None, n=n, cloud=cloud, width=width, permutation=rng.random() < 0.25,
                      autobox=rng.random() < 0.3, graph=rng.random() < 0.4,
                      tuned=n > 2000000 and rng.random() < 0.3)
    if kind == "batch":
        clouds = _log_size(rng, 3, 200)
        return {"kind": "batch", "clouds": clouds, "lo": _log_size(rng, 500, 8192),
                "hi": min(_log_size(rng, 20000, 1000000), 33000000 // clouds), "width": width,
                "graph": rng.random() < 0.5, "boxes": rng.random() < 0.6}
    if kind == "stages":
        return {"kind": "stages", "n": _log_size(rng, 3000, 8000000), "cloud": cloud,
                "width": width}
    if kind == "stream":
        return {"kind": "stream", "n": _log_size(rng, 20000, 3000000), "cloud": cloud,
                "frames": rng.randint(2, 8)}
    if kind == "sort":
        return {"kind": "sort", "n": _log_size(rng, 2000, 1 << 24), "cloud": cloud,
                "pairs": rng.random() < 0.4}
    if kind == "learned":
        return {"kind": "learned", "n": _log_size(rng, 1 << 20, 1 << 25), "cloud": "clustered"}
    return {"kind": kind, "n": _log_size(rng, 5000, 6000000), "cloud": cloud}


# ---------------------------------------------------------------- device views
class _View:
    """Device memory of a context for torch.as_tensor; keeps its owner alive."""

    def __init__(self, owner, ptr, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(count),), "typestr": typestr,
                                         "data": (int(ptr), False), "version": 2,
                                         "strides": None}


def _tensor(owner, ptr, count, typestr):
    if count <= 0:
        dtype = {"<i4": torch.int32, "|u1": torch.uint8, "<f4": torch.float32}[typestr]
        return torch.empty(0, dtype=dtype, device="cuda")
    return torch.as_tensor(_View(owner, ptr, count, typestr), device="cuda")


def _points(ctx, n, cloud, width, seed, low=MIN, size=RANGE, salt=0):
    """(DeviceArray of a cloud in the cube [low, low + size), its tensor)"""
    arr = ctx.empty((n, width), "float32")
    t = _tensor(ctx, arr.ptr, n * width, "<f4").view(n, width)
    _fill(t, cloud, seed, low, size, salt)
    torch.cuda.synchronize()
    return arr, t


def _fill(t, cloud, seed, low, size, salt=0):
    """A cloud of 1024 cells a side in the cube [low, low + size), the box
    that the pipeline reduces from it when it is given none: one point sits on
    the low corner and one at the far end. Every seed gives another frame of
    one scene: the points of octants 1 and 2 are mirrored there, all have a
    new place in their cell and a new order, and the numbers of unique keys
    and of nodes stay those of the scene, so that outputs keep their sizes."""
    n, width = t.shape
    g = torch.Generator(device="cuda").manual_seed(n * 64 + salt)
    q = (_uniform(n, g) if cloud == "uniform" else _clustered(n, g)).to(torch.int32)
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + salt)
    octant = ((q >> 9) * torch.tensor([1, 2, 4], device="cuda", dtype=torch.int32)).sum(1)
    for k in (1, 2):
        flip = torch.randint(1, 512, (3,), generator=g, device="cuda").to(torch.int32)
        q = torch.where((octant == k)[:, None], q ^ flip, q)
    cell = size / 1024.0
    place = torch.rand((n, 3), generator=g, device="cuda").mul_(0.96).add_(0.02)
    xyz = (q + place).mul_(cell).add_(low).clamp_(max=low + size / 1.0001)
    if n >= 2:
        xyz[0], xyz[1] = low, low + size / 1.0001
    t[:, :3] = xyz[torch.randperm(n, generator=g, device="cuda")]
    if width == 4:
        t[:, 3] = 0.0


def _uniform(n, g):
    return torch.rand((n, 3), generator=g, device="cuda").mul_(RANGE).clamp_(0.0, LIMIT)


def _clustered(n, g):
    """The surface scene of pipeline_amd.clouds.clustered, drawn on the GPU."""
    def rand(*shape):
        return torch.rand(shape, generator=g, device="cuda")

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    n_plane = n_cyl = round(0.4 * n)
    n_gauss = n - n_plane - n_cyl
    plane = torch.cat([rand(n_plane, 2) * RANGE, normal(n_plane, 1) * 0.5], 1)
    cen, rad, hgt = rand(32, 2) * RANGE, 2.0 + 18.0 * rand(32), 5.0 + 195.0 * rand(32)
    which = torch.randint(0, 32, (n_cyl,), generator=g, device="cuda")
    theta = rand(n_cyl) * (2.0 * math.pi)
    cyl = torch.stack([cen[which, 0] + rad[which] * torch.cos(theta),
                       cen[which, 1] + rad[which] * torch.sin(theta),
                       rand(n_cyl) * hgt[which]], 1)
    gc, gs = rand(64, 3) * RANGE, 1.0 + 29.0 * rand(64)
    which = torch.randint(0, 64, (n_gauss,), generator=g, device="cuda")
    gauss = gc[which] + normal(n_gauss, 3) * gs[which, None]
    return torch.cat([gauss, plane, cyl]).clamp_(0.0, LIMIT)


def _keys(ctx, n, cloud, seed):
    """n Morton keys of a cloud in a device array (16-byte padded)."""
    pts, _ = _points(ctx, n, cloud, 3, seed)
    keys = ctx.empty((n + 3) // 4 * 4, "uint32")
    ctx.k_ComputeMortonCode(pts, keys, n, MIN, RANGE)
    ctx.synchronize()
    pts.free()
    return keys


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    return {"frame": _prepare_frame, "batch": _prepare_batch, "stages": _prepare_stages,
            "stream": _prepare_stream, "sort": _prepare_sort, "learned": _prepare_learned,
            "compact": _prepare_compact, "expand": _prepare_expand}[case["kind"]](case, seed)


def _prepare_frame(case, seed):
    ctx = Context(0)
    if case["tuned"]:
        ctx.set_tune(**TUNED)
    ctx.set_graph_mode(case["graph"])
    ctx.set_permutation(case["permutation"])
    pts, _ = _points(ctx, case["n"], case["cloud"], case["width"], seed)
    return {"case": case, "ctx": ctx, "pts": pts, "views": None}


def _batch_sizes(case):
    """Log-uniform sizes, fixed by the case (a golden-ratio sequence)."""
    lo, hi, k = math.log(case["lo"]), math.log(max(case["hi"], case["lo"] + 1)), case["clouds"]
    return [int(math.exp(lo + (hi - lo) * ((i + 1) * 0.6180339887498949 % 1.0)))
            for i in range(k)]


def _prepare_batch(case, seed):
    ctx = Context(0)
    ctx.set_graph_mode(case["graph"])
    sizes = _batch_sizes(case)
    offs = [0]
    for s in sizes:
        offs.append(offs[-1] + s)
    w = case["width"]
    pts = ctx.empty((offs[-1], w), "float32")
    t = _tensor(ctx, pts.ptr, offs[-1] * w, "<f4").view(offs[-1], w)
    low = [-2000.0 + 4000.0 * ((k * 0.5698402909980532) % 1.0) for k in range(len(sizes))]
    size = [50.0 + 4000.0 * ((k * 0.7548776662466927) % 1.0) for k in range(len(sizes))]
    for k in range(len(sizes)):
        _fill(t[offs[k]:offs[k + 1]], "uniform" if k % 2 == 0 else "clustered", seed, low[k],
              size[k], salt=k)
    torch.cuda.synchronize()
    return {"case": case, "ctx": ctx, "pts": pts, "offs": offs, "views": None, "min": low,
            "range": size}


def _prepare_stages(case, seed):
    n = case["n"]
    ctx = Context(0)
    pts, _ = _points(ctx, n, case["cloud"], case["width"], seed)
    st = {"case": case, "ctx": ctx, "pts": pts, "views": None}
    for name, dtype in (("keys", "uint32"), ("alt", "uint32"), ("pn", "uint8"), ("hl", "uint8"),
                        ("hr", "uint8"), ("lc", "int32"), ("par", "int32"), ("edge", "int32"),
                        ("offs", "int32")):
        st[name] = ctx.zeros(n, dtype)
    st["nodes"] = ctx.zeros(n * NODE_BYTES, "uint8")
    return st


def _prepare_stream(case, seed):
    ppl = Pipeline(2, max_points=case["n"])
    ctx = ppl.context(0)
    frames = [_points(ctx, case["n"], case["cloud"], 4, seed * 3 + k)[0] for k in range(3)]
    return {"case": case, "ppl": ppl, "frames": frames, "views": {}}


def _prepare_sort(case, seed):
    ctx = Context(0)
    keys = _keys(ctx, case["n"], case["cloud"], seed)
    n = keys.size
    st = {"case": case, "ctx": ctx, "src": keys, "keys": ctx.zeros(n, "uint32"),
          "alt": ctx.zeros(n, "uint32")}
    out = [_tensor(ctx, st["keys"].ptr, case["n"], "<i4")]
    if case["pairs"]:
        for name in ("vsrc", "vals", "valt"):
            st[name] = ctx.zeros(n, "uint32")
        _tensor(ctx, st["vsrc"].ptr, n, "<i4").copy_(torch.arange(n, dtype=torch.int32))
        out.append(_tensor(ctx, st["vals"].ptr, case["n"], "<i4"))
    ctx.synchronize()
    torch.cuda.synchronize()
    st["out"] = out
    return st


def _prepare_learned(case, seed):
    ctx = Context(0)
    n = case["n"]
    keys = _keys(ctx, n, case["cloud"], seed)
    # The earlier frame: the same scene, its points moved a little, so that
    # the model knows the distribution but not these keys.
    pts, t = _points(ctx, n, case["cloud"], 3, seed)
    t.add_(0.75).clamp_(0.0, LIMIT)
    torch.cuda.synchronize()
    prev = ctx.empty(n, "uint32")
    ctx.k_ComputeMortonCode(pts, prev, n, MIN, RANGE)
    ctx.synchronize()
    ctx.cdf_reset()
    ctx.cdf_add_samples(prev, n, 100)
    ctx.cdf_train(steps=1000)
    pts.free()
    prev.free()
    st = {"case": case, "ctx": ctx, "src": keys, "keys": ctx.zeros(keys.size, "uint32"),
          "alt": ctx.zeros(keys.size, "uint32")}
    st["out"] = [_tensor(ctx, st["keys"].ptr, n, "<i4")]
    ctx.synchronize()
    return st


def _built(case, seed):
    """A context that has built the case's cloud, and its octree's size."""
    ctx = Context(0)
    pts, _ = _points(ctx, case["n"], case["cloud"], 4, seed)
    ctx.build(pts, case["n"], MIN, RANGE)
    _, k = ctx.counts(1)
    return ctx, int(k[0])


def _compact_call(st):
    """ocp_compact_octree into the state's own arrays: (nodes, children)."""
    ctx, kn, kc = st["ctx"], ctypes.c_int64(), ctypes.c_int64()
    rc = ctx.lib.ocp_compact_octree(ctx.h, st["nodes"].ptr, st["nodes"].size, st["children"].ptr,
                                    st["children"].size, ctypes.byref(kn), ctypes.byref(kc))
    if rc != pipeline_amd.OCP_OK:
        raise RuntimeError("ocp_compact_octree: status %d" % rc)
    return kn.value, kc.value


def _prepare_compact(case, seed):
    ctx, k = _built(case, seed)
    st = {"case": case, "ctx": ctx, "views": None,
          "nodes": ctx.zeros(k, pipeline_amd.COMPACT_NODE_DTYPE),
          "children": ctx.zeros(4 * case["n"] + 8, "int32")}
    ctx.synchronize()
    return st


def _prepare_expand(case, seed):
    ctx, _ = _built(case, seed)
    nodes, children = ctx.compact_octree()
    out = ctx.zeros(nodes.size * NODE_BYTES, "uint8")
    ctx.synchronize()
    return {"case": case, "ctx": ctx, "nodes": nodes, "children": children, "dst": out,
            "oct_start": ctx.results().oct_start,
            "out": [_tensor(ctx, out.ptr, out.size // 4, "<i4")]}


# ---------------------------------------------------------------- run
def run(state):
    return _RUN[state["case"]["kind"]](state)


def _run_frame(st):
    ctx, case = st["ctx"], st["case"]
    if case["autobox"]:
        ctx.build_autobox(st["pts"], case["n"])
    else:
        ctx.build(st["pts"], case["n"], MIN, RANGE)
    u, k = ctx.counts(1)
    return _frame_views(st, ctx, (int(u[0]), int(k[0])))


def _frame_views(st, ctx, size):
    """The build's outputs as tensors, made again only when a size changed
    (the buffers stay where they are between builds of one shape)."""
    kept = st["views"]
    if kept is None or kept[0] != size:
        r = ctx.results()
        n, u, k = int(r.n_points), size[0], size[1]
        m = max(u - 1, 0)
        out = [_tensor(ctx, p, c, "<i4") for p, c in (
            (r.sorted_keys, n), (r.unique_keys, u), (r.left_child, m), (r.parent, m),
            (r.edge_count, m), (r.offsets, m), (r.nodes, k * NODE_BYTES // 4))]
        out += [_tensor(ctx, p, m, "|u1") for p in (r.prefix_n, r.has_leaf_left,
                                                    r.has_leaf_right)]
        if r.sorted_index:
            out += [_tensor(ctx, r.sorted_index, n, "<i4"), _tensor(ctx, r.unique_index, u, "<i4")]
        st["views"] = kept = (size, out)
    return [size[0], size[1], kept[1]]


def _run_batch(st):
    ctx, case = st["ctx"], st["case"]
    if case["boxes"]:
        ctx.build_batched(st["pts"], st["offs"], st["min"], st["range"])
    else:
        ctx.build_batched(st["pts"], st["offs"])
    u, k = ctx.counts(case["clouds"])
    total = int(k.sum())
    if st["views"] is None:
        r = ctx.results()
        st["views"] = [_tensor(ctx, r.sorted_keys, st["offs"][-1], "<i4"),
                       _tensor(ctx, r.nodes, total * NODE_BYTES // 4, "<i4")]
    return [u, k, st["views"]]


def _run_stages(st):
    ctx, n = st["ctx"], st["case"]["n"]
    ctx.k_ComputeMortonCode(st["pts"], st["keys"], n, MIN, RANGE)
    ctx.k_SortKeys(st["keys"], st["alt"], n)
    u = ctx.k_CountUnique(st["keys"], n)
    m = u - 1
    ctx.k_BuildRadixTree(m, st["keys"], st["pn"], st["hl"], st["hr"], st["lc"], st["par"])
    ctx.k_EdgeCount(st["pn"], st["par"], st["edge"], m)
    ctx.k_PartialSum(st["edge"], 0, m, st["offs"])
    # The last offset bounds the slots: a chain has at most ten.
    last = pipeline_amd.d2h(ctx, st["offs"].ptr + 4 * (m - 1), 1, "int32")
    k = int(last[0]) + 10
    ctx.k_InitOctNodes(st["nodes"], k, st["keys"], st["pn"], m, MIN, RANGE)
    ctx.k_MakeOctNodes(st["nodes"], st["offs"], st["edge"], st["keys"], st["pn"], st["par"], MIN,
                       RANGE, m, k)
    ctx.k_LinkLeafNodes(st["nodes"], st["offs"], st["edge"], st["keys"], st["hl"], st["hr"],
                        st["pn"], st["par"], st["lc"], m, k)
    ctx.synchronize()
    if st["views"] is None:
        st["views"] = [_tensor(ctx, st["keys"].ptr, u, "<i4")]
        st["views"] += [_tensor(ctx, st[f].ptr, m, "<i4") for f in ("lc", "par", "edge", "offs")]
        st["views"] += [_tensor(ctx, st[f].ptr, m, "|u1") for f in ("pn", "hl", "hr")]
        st["views"].append(_tensor(ctx, st["nodes"].ptr, k * NODE_BYTES // 4, "<i4"))
    return [u, st["views"]]


def _run_stream(st):
    ppl, case = st["ppl"], st["case"]
    for f in range(case["frames"]):
        if f >= 2:
            ppl.wait(f % 2)
        ppl.submit(f % 2, st["frames"][f % 3], case["n"])
    out = []
    for slot in range(2):
        ppl.wait(slot)
        u, k = ppl.context(slot).counts(1)
        kept = st["views"].setdefault(slot, {"views": None, "ppl": ppl})
        out.append(_frame_views(kept, _Slot(ppl, slot), (int(u[0]), int(k[0]))))
    return out


class _Slot:
    """A slot's context that keeps its pipeline alive in the views."""

    def __init__(self, ppl, slot):
        self.ppl, self.slot = ppl, slot

    def results(self):
        return self.ppl.context(self.slot).results()


def _run_sort(st):
    ctx, n, size = st["ctx"], st["case"]["n"], st["src"].nbytes
    ctx.copy(st["keys"], st["src"], size)
    if st["case"]["pairs"]:
        ctx.copy(st["vals"], st["vsrc"], size)
        ctx.k_SortPairs(st["keys"], st["vals"], st["alt"], st["valt"], n)
    else:
        ctx.k_SortKeys(st["keys"], st["alt"], n)
    ctx.synchronize()
    return st["out"]


def _run_learned(st):
    ctx = st["ctx"]
    ctx.copy(st["keys"], st["src"], st["src"].nbytes)
    ctx.sort_learned(st["keys"], st["alt"], st["case"]["n"])
    return st["out"]


def _run_compact(st):
    kn, kc = _compact_call(st)
    if st["views"] is None:
        ctx = st["ctx"]
        st["views"] = [_tensor(ctx, st["nodes"].ptr, 3 * kn, "<i4"),
                       _tensor(ctx, st["children"].ptr, st["children"].size, "<i4")]
    return [kn, kc, st["views"]]


def _run_expand(st):
    ctx = st["ctx"]
    rc = ctx.lib.ocp_expand_octree(ctx.h, st["nodes"].ptr, st["children"].ptr,
                                   st["children"].size, ctypes.c_void_p(st["oct_start"]), 1, None,
                                   None, MIN, RANGE, st["dst"].ptr)
    if rc != pipeline_amd.OCP_OK:
        raise RuntimeError("ocp_expand_octree: status %d" % rc)
    ctx.synchronize()
    return st["out"]


_RUN = {"frame": _run_frame, "batch": _run_batch, "stages": _run_stages, "stream": _run_stream,
        "sort": _run_sort, "learned": _run_learned, "compact": _run_compact,
        "expand": _run_expand}


# ---------------------------------------------------------------- work
def _tree_sizes(n, cloud):
    """About how many unique keys and octree nodes n points give: uniform
    points fall into 2^30 cells; clustered ones share keys on their surfaces.
    Half a node per unique key in the mean over sizes."""
    cells = float(1 << 30) if cloud == "uniform" else 1.2e7
    u = cells * -math.expm1(-n / cells)
    return u, 0.5 * u


def _build_bytes(n, cloud, width, permutation=False):
    """Points read, every stage output written once."""
    u, k = _tree_sizes(n, cloud)
    b = 4.0 * width * n + 4.0 * n + 4.0 * u + 19.0 * u + NODE_BYTES * k
    return b + 4.0 * (n + u) if permutation else b


def work(case):
    kind = case["kind"]
    if kind == "batch":
        b = sum(_build_bytes(s, "uniform" if k % 2 == 0 else "clustered", case["width"])
                for k, s in enumerate(_batch_sizes(case)))
    elif kind == "frame":
        b = _build_bytes(case["n"], case["cloud"], case["width"], case["permutation"])
    elif kind == "stages":
        b = _build_bytes(case["n"], case["cloud"], case["width"])
    elif kind == "stream":
        b = case["frames"] * _build_bytes(case["n"], case["cloud"], 4)
    elif kind in ("sort", "learned"):
        b = 8.0 * case["n"] * (2 if case.get("pairs") else 1)
    else:  # 60-byte nodes on one side; 12-byte nodes and the child indices on the other
        u, k = _tree_sizes(case["n"], case["cloud"])
        b = (NODE_BYTES + 12.0) * k + 4.0 * (u + k)
    return {"bytes": b, "flops": 0.0}


def exact(case, seed):
    return None
