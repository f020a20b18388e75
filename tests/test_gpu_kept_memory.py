"""The device memory that the engine keeps between calls: blocks of released dense buffers and
the workspace of calls on the engine stream.

Bar: bit for bit what the same call gives on memory of its own. Calls write into blocks that
queued work has just used, sizes on both sides of a block class and above the largest one,
workspaces grow between calls, and calls on a stream of the caller's run beside calls on the
engine stream.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from jax4j_amd import DType, QuantType
from jax4j_amd import _native as N
from jax4j_amd import synthetic as S

pytestmark = pytest.mark.gpu


def upload(backend, qt, rows, cols, seed):
    return backend.upload_quantized(S.quant_blocks(qt, seed, rows, cols), qt, (rows, cols))


# 64 and 65 floats: both sides of a 256-byte block; 1 Mi and 1 Mi + 32: of the largest (4 MiB)
@pytest.mark.parametrize("rows", [1, 64, 65, 4096, 1 << 20, (1 << 20) + 32])
def test_results_in_reused_blocks_are_those_of_fresh_ones(backend, rows):
    w = upload(backend, QuantType.Q4_0, rows, 32, 5)
    xs = [backend.upload(S.activations_f32(7 + i, 32)) for i in range(3)]
    keep = [backend.quant_matvec(w, x) for x in xs]
    fresh = [backend.download(y) for y in keep]
    for i in range(12):  # each result's block goes to the next call while its work may be queued
        y = backend.quant_matvec(w, xs[i % 3])
        z = backend.quant_matvec_add(w, xs[(i + 1) % 3], y)
        backend.release(y)
        g = backend.quant_gather_row(w, rows - 1)
        backend.release(g)
        got = backend.download(z)
        assert np.array_equal(got.view(np.uint32), (fresh[(i + 1) % 3] + fresh[i % 3]).view(np.uint32))
        backend.release(z)
    for b in [w, *xs, *keep]:
        backend.release(b)


class Hip:
    """The HIP runtime the engine is linked to: a stream of the caller's, and stream capture."""

    def __init__(self):
        self.lib = N.load()
        self.stream = C.c_void_p()
        self.ok("hipStreamCreateWithFlags", C.byref(self.stream), 1)  # non-blocking

    def ok(self, name, *args):
        assert getattr(self.lib, name)(*args) == 0, name

    def wait(self):
        self.ok("hipDeviceSynchronize")

    def close(self):
        self.wait()
        self.ok("hipStreamDestroy", self.stream)


def test_an_address_given_out_is_not_reused_behind_its_work(backend):
    """A buffer whose address was read may be in use on a stream of the caller's when it is released:
    the work queued there still sees its own values."""
    n = 1 << 18
    hip, lib = Hip(), N.load()
    values = S.activations_f32(11, n)
    b, out = backend.upload(values), backend.upload(np.zeros(n, np.float32))
    src, dst = (backend.buffer_desc(h).device_ptr for h in (b, out))
    assert lib.j4q_spin(3000, hip.stream) == 0
    assert lib.j4q_copy(dst, src, 4 * n, hip.stream) == 0
    backend.release(b)
    others = [backend.upload(np.full(n, np.nan, np.float32)) for _ in range(2)]
    hip.wait()
    assert np.array_equal(backend.download(out), values)
    for h in [out, *others]:
        backend.release(h)
    hip.close()


@pytest.mark.parametrize("qt", [QuantType.Q4_K, QuantType.Q8_0], ids=lambda q: q.name)
def test_workspace_calls_on_two_streams_and_growing(backend, qt):
    """16 rows over several column windows use a workspace: one kept for the engine stream that grows
    from the first matrix to the second, stream-ordered memory on another stream."""
    hip = Hip()
    shapes = [(96, 4096), (4000, 8192)]
    ws = [upload(backend, qt, r, k, 20 + r) for r, k in shapes]
    xs = [backend.upload(S.activations_f32(3 + k, 16 * k), shape=(16, k)) for _, k in shapes]
    ptr = lambda h: backend.buffer_desc(h).device_ptr

    def result(i):
        return backend.upload(np.full((16, shapes[i][0]), np.nan, np.float32))

    def call(i, y, stream):
        backend.quant_matvec_into(ws[i], ptr(xs[i]), 0, ptr(y), 16, stream)

    ref = []
    for i in range(2):  # alone, each waited for
        y = result(i)
        call(i, y, hip.stream.value)
        hip.wait()
        ref.append(backend.download(y))
        backend.release(y)
    calls = [(0, 0), (1, hip.stream.value), (1, 0), (0, hip.stream.value), (0, 0), (1, 0)]
    ys = [result(i) for i, _ in calls]
    for (i, stream), y in zip(calls, ys):
        call(i, y, stream)
    hip.wait()
    for (i, _), y in zip(calls, ys):
        assert np.array_equal(backend.download(y).view(np.uint32), ref[i].view(np.uint32))
    for h in [*ws, *xs, *ys]:
        backend.release(h)
    hip.close()


# 24 rows over 1024 columns: a call that runs in 16-row launches under capture, and needs no workspace there
@pytest.mark.parametrize("b,r,k", [(16, 640, 4096), (24, 640, 1024)])
def test_workspace_call_under_capture_replays(backend, b, r, k):
    """Under capture of the engine stream a call takes memory of the graph, not the kept workspace: eager
    calls between the replays do not change what they give."""
    hip = Hip()
    st = C.c_void_p(backend.stream())
    w = upload(backend, QuantType.Q4_K, r, k, 31)
    x = backend.upload(S.activations_f32(5, b * k), shape=(b, k))
    y, z = (backend.upload(np.zeros((b, r), np.float32)) for _ in range(2))
    px, py, pz = (backend.buffer_desc(h).device_ptr for h in (x, y, z))
    nan = backend.upload(np.full((b, r), np.nan, np.float32))
    pnan = backend.buffer_desc(nan).device_ptr
    for b0 in range(0, b, 16):
        backend.quant_matvec_into(w, px + 4 * b0 * k, 0, pz + 4 * b0 * r, min(16, b - b0))
    ref = backend.download(z).view(np.uint32)
    graph, run = C.c_void_p(), C.c_void_p()
    hip.ok("hipStreamBeginCapture", st, 2)  # relaxed
    backend.quant_matvec_into(w, px, 0, py, b)
    hip.ok("hipStreamEndCapture", st, C.byref(graph))
    hip.ok("hipGraphInstantiate", C.byref(run), graph, None, None, C.c_size_t(0))
    for _ in range(4):
        assert N.load().j4q_copy(py, pnan, 4 * b * r, None) == 0
        hip.ok("hipGraphLaunch", run, st)
        backend.quant_matvec_into(w, px, 0, pz, b)
        assert np.array_equal(backend.download(y).view(np.uint32), ref)
        if b == 16:
            assert np.array_equal(backend.download(z).view(np.uint32), ref)
    hip.ok("hipGraphExecDestroy", run)
    hip.ok("hipGraphDestroy", graph)
    for h in (w, x, y, z, nan):
        backend.release(h)
    hip.close()


def test_captured_matmul_replays(backend):
    """A GEMM that splits K over a workspace when called does not under capture: the same products in another
    order of their fp32 sums, on every replay."""
    m, n, k = 24, 512, 8192
    hip = Hip()
    w = upload(backend, QuantType.Q6_K, n, k, 51)
    x = backend.upload(S.activations_bf16(9, m * k).reshape(m, k), shape=(m, k), dtype=DType.BF16)
    y, z, nan = (backend.upload(np.full((m, n), np.nan, np.float32)) for _ in range(3))
    px, py, pz, pnan = (backend.buffer_desc(h).device_ptr for h in (x, y, z, nan))
    graph, runs = C.c_void_p(), [C.c_void_p(), C.c_void_p()]
    hip.ok("hipStreamBeginCapture", hip.stream, 2)  # relaxed
    backend.quant_matmul_into(w, px, m, "bf16", 0, 0, py, hip.stream.value)
    hip.ok("hipStreamEndCapture", hip.stream, C.byref(graph))
    for run in runs:  # a graph without memory nodes may be instantiated more than once
        hip.ok("hipGraphInstantiate", C.byref(run), graph, None, None, C.c_size_t(0))
    first = None
    for i in range(4):
        assert N.load().j4q_copy(py, pnan, 4 * m * n, hip.stream) == 0
        hip.ok("hipGraphLaunch", runs[i % 2], hip.stream)
        backend.quant_matmul_into(w, px, m, "bf16", 0, 0, pz)
        hip.wait()
        got, eager = backend.download(y), backend.download(z)
        first = got if first is None else first
        assert np.array_equal(got.view(np.uint32), first.view(np.uint32))
        assert np.abs(got - eager).max() <= 4e-5 * np.abs(eager).max()  # each within 2e-5 of the exact sums
    for run in runs:
        hip.ok("hipGraphExecDestroy", run)
    hip.ok("hipGraphDestroy", graph)
    for h in (w, x, y, z, nan):
        backend.release(h)
    hip.close()


def test_workspaces_of_many_streams(backend):
    """Streams that take a workspace over from another, one whose work is still queued among them, and one
    created where another was destroyed: every result is that of a call alone."""
    b, shapes = 40, [(700, 1024), (4000, 2048)]
    lib = N.load()
    ws = [upload(backend, QuantType.Q6_K, r, k, 40 + r) for r, k in shapes]
    xs = [backend.upload(S.activations_f32(6 + k, b * k), shape=(b, k)) for _, k in shapes]
    ptr = lambda h: backend.buffer_desc(h).device_ptr
    ref = []
    for w, x in zip(ws, xs):
        y = backend.quant_matvec(w, x)
        ref.append(backend.download(y).view(np.uint32))
        backend.release(y)
    hips = [Hip() for _ in range(3)]
    results = []

    def call(i, hip):
        y = backend.upload(np.full((b, shapes[i][0]), np.nan, np.float32))
        results.append((i, y))
        backend.quant_matvec_into(ws[i], ptr(xs[i]), 0, ptr(y), b, hip.stream.value)

    for turn in range(4):
        for k, hip in enumerate(hips):
            assert lib.j4q_spin(200 * ((k + turn) % 3), hip.stream) == 0
            call((k + turn) % 2, hip)
            call((k + turn + 1) % 2, hip)
        hips[turn % 3].ok("hipStreamDestroy", hips[turn % 3].stream)  # its calls are still queued
        hips[turn % 3] = Hip()
        call(turn % 2, hips[turn % 3])
    for hip in hips:
        hip.close()
    for i, y in results:
        assert np.array_equal(backend.download(y).view(np.uint32), ref[i])
    for h in [*ws, *xs, *(y for _, y in results)]:
        backend.release(h)


# 1 row: no workspace; 24 rows: tiles, the event on the GEMV's launch; 16 rows: on the window sums'
@pytest.mark.parametrize("handle", [1, 2], ids=["hipStreamLegacy", "hipStreamPerThread"])
@pytest.mark.parametrize("qt,b,r,k", [(QuantType.Q8_0, 1, 640, 1024), (QuantType.Q8_0, 24, 1000, 1024), (QuantType.Q4_K, 16, 640, 4096)])
def test_workspaces_on_the_runtimes_own_streams(backend, handle, qt, b, r, k):
    """The runtime's two stream handles that name no stream object of their own."""
    hip = Hip()
    w = upload(backend, qt, r, k, 61)
    x = backend.upload(S.activations_f32(3, b * k), shape=(b, k))
    ref = backend.quant_matvec(w, x)
    y = backend.upload(np.full((b, r), np.nan, np.float32))
    px, py = (backend.buffer_desc(h).device_ptr for h in (x, y))
    print("[case]", qt.name, b, r, k, "stream handle", handle, flush=True)
    for _ in range(3):
        backend.quant_matvec_into(w, px, 0, py, b, handle)
    hip.wait()
    assert np.array_equal(backend.download(y).view(np.uint32).reshape(-1), backend.download(ref).view(np.uint32).reshape(-1))
    for h in (w, x, ref, y):
        backend.release(h)
    hip.close()


@pytest.mark.parametrize("handle", [1, 2], ids=["hipStreamLegacy", "hipStreamPerThread"])
def test_matmul_workspaces_on_the_runtimes_own_streams(backend, handle):
    m, n, k = 24, 512, 8192  # K split, the event on the sums' launch
    hip = Hip()
    w = upload(backend, QuantType.Q6_K, n, k, 51)
    x = backend.upload(S.activations_bf16(9, m * k).reshape(m, k), shape=(m, k), dtype=DType.BF16)
    ref = backend.quant_matmul(w, x, "bf16")
    y = backend.upload(np.full((m, n), np.nan, np.float32))
    px, py = (backend.buffer_desc(h).device_ptr for h in (x, y))
    for _ in range(3):
        backend.quant_matmul_into(w, px, m, "bf16", 0, 0, py, handle)
    hip.wait()
    assert np.array_equal(backend.download(y).view(np.uint32), backend.download(ref).view(np.uint32))
    for h in (w, x, ref, y):
        backend.release(h)
    hip.close()
