"""Calls recorded into a caller's own graph on the context's stream, replayed
among the program's eager builds, whose sort may have changed its form since."""
import ctypes

import numpy as np
import pytest

import oracle
import pipeline_amd
from pipeline_amd import Context
from test_gpu_pipeline import _check_segment
from test_gpu_tree_tiles import _cells

pytestmark = pytest.mark.gpu


class _Capture:
    """A context on a stream of the test's, and graphs of its calls."""

    def __init__(self):
        self.hip = ctypes.CDLL("libamdhip64.so")
        self.stream, h = ctypes.c_void_p(), ctypes.c_void_p()
        self._ok(self.hip.hipStreamCreate(ctypes.byref(self.stream)))
        lib = pipeline_amd.load_library()
        assert lib.ocp_create(ctypes.byref(h), 0, self.stream) == pipeline_amd.OCP_OK
        self.ctx = Context.__new__(Context)
        self.ctx.lib, self.ctx.h, self.ctx._owned = lib, h, []
        self.graphs = []

    def _ok(self, rc):
        assert rc == 0, f"HIP status {rc}"

    def record(self, call):
        graph, ex = ctypes.c_void_p(), ctypes.c_void_p()
        self._ok(self.hip.hipStreamBeginCapture(self.stream, 1))  # thread-local
        call()
        self._ok(self.hip.hipStreamEndCapture(self.stream, ctypes.byref(graph)))
        self._ok(self.hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None,
                                              ctypes.c_size_t(0)))
        self._ok(self.hip.hipGraphDestroy(graph))
        self.graphs.append(ex)
        return lambda: self._ok(self.hip.hipGraphLaunch(ex, self.stream))

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.ctx.close()
        for ex in self.graphs:
            self._ok(self.hip.hipGraphExecDestroy(ex))
        self._ok(self.hip.hipStreamDestroy(self.stream))


def test_batch_whose_sort_changes_its_form():
    """Crowded keys: once the counts are read, builds of this size take another
    sort. A graph recorded before and one recorded after that both stay right."""
    rng = np.random.default_rng(8)
    sizes = [30_000, 20_001, 9000]
    pts = [_cells((700 << 20) + rng.integers(0, 1 << 18, s)) for s in sizes]
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    exp = [oracle.build_plain(p) for p in pts]
    with _Capture() as cap:
        ctx = cap.ctx
        d = ctx.upload(np.concatenate(pts))

        def build():
            ctx.build_batched(d, offs, [0.0] * 3, [1024.0] * 3)

        def check():
            out = ctx.fetch(offs)
            for k in range(3):
                _check_segment(out, k, exp[k])
        build()
        first = cap.record(build)
        build()
        check()  # (reads the counts)
        second = cap.record(build)
        for _ in range(3):
            for replay in (first, second):
                replay()
                check()
                build()
                check()


def test_replayed_time_out_is_reported():
    """A wait that gives up in a replay, after a build whose report was good."""
    rng = np.random.default_rng(3)
    keys = rng.integers(0, 1 << 30, 300_000, dtype=np.uint32)
    pts = _cells(rng.integers(0, 1 << 30, 20_000))
    with _Capture() as cap:
        ctx = cap.ctx
        d, alt, p = ctx.upload(keys), ctx.empty(keys.size, np.uint32), ctx.upload(pts)
        ctx.k_SortKeys(d, alt, keys.size)
        ctx.synchronize()
        replay = cap.record(lambda: ctx.k_SortKeys(d, alt, keys.size))
        for limit in (-1, 0, -1):
            d.copy_from(keys)
            ctx.set_wait_limit(-1)
            ctx.build(p, pts.shape[0], 0.0, 1024.0)
            ctx.synchronize()
            ctx.set_wait_limit(limit)
            replay()
            if limit == 0:
                with pytest.raises(pipeline_amd.OcpError, match="wait gave up"):
                    ctx.synchronize()
            else:
                ctx.synchronize()
                np.testing.assert_array_equal(d.to_host(), np.sort(keys))
                ctx.counts(1)
