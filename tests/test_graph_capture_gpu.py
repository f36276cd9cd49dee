"""Library calls recorded in a caller's HIP graph (GPU).

The graph may be replayed beside the library stream, so recorded calls keep off
the static memory that launches on that stream share (gemm_partials of
mxh_internal.h): it holds a pattern here that every replay must leave.  Replays
on another stream, with eager work between them, against eager results.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import mxhip
import mxo
from test_attention_prefill_gpu import reference

pytestmark = pytest.mark.gpu


class Graph:
    """What `calls` launch on the library stream, recorded and replayed on a stream of its own."""

    def __init__(self, calls):
        self.hip = C.CDLL("libamdhip64.so.7")  # the runtime the library has loaded
        lib, self.stream, self.exe = C.c_void_p(mxhip.lib.mxh_stream()), C.c_void_p(), C.c_void_p()
        graph = C.c_void_p()
        mxhip.synchronize()
        self.ok(self.hip.hipStreamCreateWithFlags(C.byref(self.stream), 1))
        self.ok(self.hip.hipStreamBeginCapture(lib, 1))  # thread-local
        for f in calls:
            f()
        self.ok(self.hip.hipStreamEndCapture(lib, C.byref(graph)))
        self.ok(self.hip.hipGraphInstantiate(C.byref(self.exe), graph, None, None, 0))
        self.ok(self.hip.hipGraphDestroy(graph))

    def ok(self, rc):
        assert rc == 0, f"HIP status {rc}"

    def replay(self):
        self.ok(self.hip.hipGraphLaunch(self.exe, self.stream))
        self.ok(self.hip.hipStreamSynchronize(self.stream))

    def close(self):
        self.ok(self.hip.hipGraphExecDestroy(self.exe))
        self.ok(self.hip.hipStreamDestroy(self.stream))


def shared_workspace():
    f = getattr(mxhip.lib, "_ZN3mxh13gemm_partialsEPm")
    f.restype, f.argtypes = C.c_void_p, [C.POINTER(C.c_size_t)]
    n = C.c_size_t()
    return f(C.byref(n)), n.value


def test_recorded_calls_leave_the_shared_workspace(mxh):
    lib, rng = mxhip.lib, np.random.default_rng(5)
    # a GEMM that splits K, and few queries over many keys
    m, n, k = 40, 512, 8192
    w = mxo.quantize(mxo.Q8_0, rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02))
    a = rng.standard_normal((m, k), dtype=np.float32)
    nh, nkv, hd, p0, rows = 8, 2, 64, 3000, 5
    q = rng.standard_normal((rows, nh * hd)).astype(np.float32)
    kc, vc = (rng.standard_normal((p0 + rows, nkv * hd)).astype(np.float16) for _ in range(2))
    dw, da, dq, dk, dv = (mxhip.DeviceBuffer.from_array(x) for x in (w, a, q, kc, vc))
    out, out2, att = (mxhip.DeviceBuffer(4 * c) for c in (m * n, m * n, rows * nh * hd))

    def noalloc():
        mxhip.check(lib.mxh_gemm_q_f16_noalloc(mxo.Q8_0, da.ptr, m, dw.ptr, n, k, out.ptr, 0), "noalloc")

    def gemm():
        mxhip.check(lib.mxh_gemm_q_f16(mxo.Q8_0, da.ptr, m, dw.ptr, n, k, out2.ptr, 0), "gemm")

    def attention():
        mxhip.check(lib.mxh_attention_prefill(dq.ptr, dk.ptr, dv.ptr, att.ptr, p0, rows, nh, nkv, hd), "attention")

    def results():
        mxhip.synchronize()
        return [b.download(np.float32, c) for b, c in ((out, m * n), (out2, m * n), (att, rows * nh * hd))]

    for f in (noalloc, gemm, attention):
        f()
    eager = results()
    want = reference(q, kc, vc, p0, rows, nh, nkv, hd).reshape(-1)
    graph = Graph([noalloc, gemm, attention])
    at, size = shared_workspace()
    pattern = np.full(size, 0xA5, np.uint8)
    for _ in range(3):
        assert lib.mxh_upload(at, pattern.ctypes.data, size) == 0
        for b in (out, out2, att):
            mxhip.check(lib.mxh_memset(b.ptr, 0xFF, b.nbytes), "memset")
        mxhip.synchronize()
        graph.replay()
        got, after = results(), np.empty(size, np.uint8)
        assert lib.mxh_download(after.ctypes.data, at, size) == 0
        assert np.array_equal(after, pattern), "a recorded call wrote to the library stream's workspace"
        assert np.array_equal(got[0], eager[0]) and np.array_equal(got[1], eager[0])
        assert np.all(np.abs(got[2] - want) <= 1e-4 * np.abs(vc.astype(np.float64)).max() + 1e-4 * np.abs(want))
        for f in (attention, gemm, noalloc):  # eager calls between the replays
            f()
        assert all(np.array_equal(x, y) for x, y in zip(results(), eager))
    graph.close()
    for b in (dw, da, dq, dk, dv, out, out2, att):
        b.close()
