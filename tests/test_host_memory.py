"""What engine calls do with device memory, on a HIP runtime that logs the calls (fakehip.py): which
memory they take, keep, give back and refuse to go without."""
from __future__ import annotations

import pytest

import fakehip


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    return fakehip.build_shim(tmp_path_factory.mktemp("fake_hip"))


@pytest.mark.parametrize("call", [
    "be.quant_matvec(w, x); operands = [x]",
    "be.quant_matvec_add(w, x, a); operands = [x, a]",
    "be.quant_matmul(w, xb, 'bf16'); operands = [xb]",
    "be.quant_matmul(w, xb, 'int8'); operands = [xb]",
    "be.quantize_act(xb); operands = [xb]",
])
def test_operands_of_a_captured_call_are_not_reused(shim, call):
    """A graph that was captured on the engine stream may run on any other: memory that it reads goes back
    with hipFree, which waits for it, and not to the engine's next result."""
    freed, reused = fakehip.run(shim, f"""
        w = zeros(QuantType.Q8_0, 64, 512)
        x, a = be.upload(np.zeros(512, np.float32)), be.upload(np.zeros(64, np.float32))
        xb = be.upload(np.zeros((8, 512), np.uint16), dtype=DType.BF16)
        fake.fake_capture(be.stream(), 1)
        {call}
        fake.fake_capture(be.stream(), 0)
        log()
        for b in operands:
            be.release(b)
        freed = len(log("free")) - len(operands)
        for n in (512, 64, 8 * 256):
            be.upload(np.zeros(n, np.float32))
        result = freed, 3 - len(log("malloc"))
    """)
    assert (freed, reused) == (0, 0)


def test_operands_of_other_calls_are_reused(shim):
    freed, taken = fakehip.run(shim, """
        w = zeros(QuantType.Q8_0, 64, 512)
        x = be.upload(np.zeros(512, np.float32))
        y = be.quant_matvec(w, x)
        log()
        be.release(x)
        be.upload(np.zeros(512, np.float32))
        result = len(log("free")), len(log("malloc"))
    """)
    assert (freed, taken) == (0, 0)


MIB = 1 << 20


@pytest.mark.parametrize("stream", ["be.stream()", "0x77770"])
def test_kept_memory_is_given_back_before_a_workspace_is_refused(shim, stream):
    """A call that needs a workspace has it as long as what is free and what the engine keeps suffice."""
    ok, refused = fakehip.run(shim, f"""
        w = zeros(QuantType.Q4_K, 512, 14336)
        x, y = address(24 * 14336 * 2), address(24 * 512 * 4)
        log()
        be.quant_matmul_into(w, x, 24, "bf16", 0, 0, y, {stream})
        need = max(int(l.split()[1]) for l in log("malloc", "malloc_async"))
        assert need <= {MIB}
        held = [be.upload(np.zeros(1 << 18, np.float32)) for _ in range(8)]
        for b in held:
            be.release(b)  # 8 MiB of blocks
        fake.fake_capacity(fake.fake_used() + 4096)
        be.quant_matmul_into(w, address(64 * 14336 * 2), 64, "bf16", 0, 0, address(64 * 512 * 4), {stream})
        assert max(int(l.split()[1]) for l in log("malloc", "malloc_async")) > {MIB}
        fake.fake_capacity(0)
        try:
            be.quant_matmul_into(w, address(640 * 14336 * 2), 640, "bf16", 0, 0, address(640 * 512 * 4), 0x99990)
            refused = None
        except RuntimeError as e:
            refused = str(e)
        result = True, refused
    """)
    assert ok and "out of memory" in refused and "workspace" in refused


CALLS = {
    "matvec": ("zeros(QuantType.Q8_0, 1000, 1024)", "lambda s: be.quant_matvec_into(w, address(4 * 24 * 1024), 0, address(4 * 24 * 1000), 24, s)"),
    "matvec of several windows": ("zeros(QuantType.Q4_K, 640, 4096)", "lambda s: be.quant_matvec_into(w, address(4 * 16 * 4096), 0, address(4 * 16 * 640), 16, s)"),
    "matmul": ("zeros(QuantType.Q6_K, 512, 4096)", "lambda s: be.quant_matmul_into(w, address(2 * 64 * 4096), 64, 'bf16', 0, 0, address(4 * 64 * 512), s)"),
}


@pytest.mark.parametrize("name", CALLS)
@pytest.mark.parametrize("done", [0, 1])
def test_calls_on_a_callers_stream_keep_their_workspace(shim, name, done):
    """From the second call on a stream takes no memory, whether the first is done or not, and the last
    launch completes the event that the next user of the workspace waits for."""
    make, call = CALLS[name]
    first, again, waits, last, other, freed = fakehip.run(shim, f"""
        w, call = {make}, {call}
        fake.fake_events_done({done})
        log()
        call(0x77770)
        first = log()
        call(0x77770)
        again = log()
        call(0x88880)  # another stream, at the same time or later
        other = log("malloc", "malloc_async", "wait")
        call(0)
        call(0)
        be.release(w)
        freed = len(log("free"))
        result = (len([l for l in first if l.startswith("malloc ")]), len([l for l in again if "alloc" in l or "free" in l]),
                  [l.split()[1] for l in again if l.startswith("wait")], again[-1].split()[-1], other, freed)
    """)
    assert first == 1 and again == 0
    assert waits == [last]  # the launch's own event, waited for by the call itself
    assert ["malloc" in l for l in other if "malloc" in l] == ([] if done else [True])
    assert [l.split()[1] for l in other if "wait" in l] != ([last] if not done else [])
    assert freed == 2 + (not done) + 1  # with the engine stream's own, and the matrix


def test_a_workspace_grows_without_a_wait_for_the_device(shim):
    """Calls return without synchronising, so a larger one leaves the smaller workspace to later calls."""
    calls, kept, bound = fakehip.run(shim, """
        w = zeros(QuantType.Q8_0, 1000, 1024)
        fake.fake_events_done(0)
        log()
        for s in (0, 0x77770):
            for b in (24, 256, 24):
                be.quant_matvec_into(w, address(4 * b * 1024), 0, address(4 * b * 1000), b, s)
        calls = log("malloc", "free", "malloc_async", "device_synchronize")
        for i in range(400):  # ever more streams, none of them done: the rest take stream-ordered memory
            be.quant_matvec_into(w, address(4 * 256 * 1024), 0, address(4 * 256 * 1000), 256, 0x100000 + 16 * i)
        used = fake.fake_used()
        many = log("malloc_async")
        be.release(w)
        result = calls, used, len(many)
    """)
    assert len(calls) == 4 and all(c.startswith("malloc ") and c.endswith("ok") for c in calls)
    assert kept <= (512 << 20) + (16 << 20) and bound > 0


@pytest.mark.parametrize("cols,nodes", [(1024, False), (2048, False), (4096, True)])
def test_captured_batches_take_memory_nodes_only_where_16_row_launches_do(shim, cols, nodes):
    got, tiles = fakehip.run(shim, f"""
        w = zeros(QuantType.Q6_K, 640, {cols})
        fake.fake_capture(0x77770, 1)
        log()
        be.quant_matvec_into(w, address(4 * 24 * {cols}), 0, address(4 * 24 * 640), 24, 0x77770)
        lines = log("malloc", "malloc_async", "launch")
        result = any("malloc" in l for l in lines), any("gemv_tile" in l for l in lines)
    """)
    assert got == nodes and tiles == nodes


# 24 rows of Q8_0 over 1024 columns (one window of 16-row launches) and over 4096, and 16 rows over 4096
@pytest.mark.parametrize("batch,cols,smaller", [(24, 1024, False), (24, 4096, True), (16, 4096, False)])
def test_batches_run_without_memory_for_a_workspace(shim, batch, cols, smaller):
    kernels, kernels_some, in_place = fakehip.run(shim, f"""
        w = zeros(QuantType.Q8_0, 640, {cols})
        x, y = address(4 * {batch * cols}), address(4 * {batch} * 640)
        def names(add, free):
            fake.fake_capacity(fake.fake_used() + free)
            log()
            be.quant_matvec_into(w, x, add, y, {batch}, 0x77770)
            return [l.split()[1] for l in log("launch")]
        result = names(0, 0), names(0, 2 * 16 * 640 * 4), names(y, 0)
    """)
    assert kernels and all("gemv_mfma" in k or "gemv_kernel" in k for k in kernels)  # no sum of windows
    assert any("sum_windows" in k for k in kernels_some) == (cols > 2048)
    assert not any("gemv_tile" in k for k in kernels + kernels_some + in_place) and in_place


def test_a_batch_that_needs_its_workspace_reports_the_missing_memory(shim):
    message, code = fakehip.run(shim, """
        w = zeros(QuantType.Q8_0, 64, 40960)
        x, y = address(4 * 24 * 40960), address(4 * 24 * 64)
        fake.fake_capacity(0)
        code = lib.j4q_quant_matvec_into(w.handle, x, y, y, 24, None)
        result = N.last_error(), code
    """)
    assert code == 5 and "out of memory" in message  # J4Q_ENOMEM


@pytest.mark.parametrize("batch", [12, 16, 30, 40])
def test_decode_plans_are_made_with_the_memory_of_16_row_launches(shim, batch):
    """Where there is no memory for more, a plan runs its sums as launches of their own and its batches in
    launches of 16 rows."""
    full, small, jobs = fakehip.run(shim, f"""
        d, kv, ffn, b = 4096, 1024, 4096, {batch}
        z = lambda r, c: zeros(QuantType.Q4_K, r, c)
        layers = [dict(q=z(d, d), k=z(kv, d), v=z(kv, d), o=z(d, d), gate=z(ffn, d), up=z(ffn, d), down=z(d, ffn)) for _ in range(2)]
        io = dict(h=address(4 * b * d), x_o=address(4 * b * d), x_down=address(4 * b * ffn), qkv=address(8 * b * (d + 2 * kv)),
                  gate_up=address(16 * b * ffn), logits=0)
        log()
        plan = be.decode_plan(layers, None, b, io)
        full = [l.split()[1] for l in log("launch")]
        size = plan.info()["plan_bytes"]
        plan.destroy()
        fake.fake_capacity(fake.fake_used() + size - 4096)
        log()
        plan = be.decode_plan(layers, None, b, io)
        small = [l.split()[1] for l in log("launch")]
        assert plan.info()["plan_bytes"] < size
        # a job's launches are kernels whose last argument's condition holds
        result = len(full), len(small), [sum("Lb1EEEvNS_4QMat" in k for k in ks) for ks in (full, small)]
    """)
    assert small > full
    assert jobs[1] == 0 and (jobs[0] > 0) == (batch <= 16)


@pytest.mark.parametrize("m,rows,cols", [(24, 512, 14336), (16, 1024, 4096), (508, 1474, 14080)])
def test_captured_matmuls_take_no_memory_nodes(shim, m, rows, cols):
    eager, captured = fakehip.run(shim, f"""
        w = zeros(QuantType.Q4_K, {rows}, {cols})
        call = lambda: lib.j4q_quant_matmul_into(w.handle, 4096, {m}, 1, None, None, 4096, 0x77770)
        log()
        assert call() == 0
        eager = log("malloc", "malloc_async", "launch")
        fake.fake_capture(0x77770, 1)
        assert call() == 0
        result = eager, log("malloc", "malloc_async", "launch")
    """)
    assert len(eager) == 3 and "sum_splits" in eager[-1]
    assert len(captured) == 1 and "gemm_tile" in captured[0]


def test_addresses_are_integers(shim):
    """Host objects whose address ctypes would pass on are refused, as pointers to GPU memory."""
    refused, launched = fakehip.run(shim, """
        w = zeros(QuantType.Q8_0, 64, 512)
        x, y = address(4 * 512), address(4 * 64)
        refused = 0
        log()
        for bad in (b"x" * 2048, "x", (C.c_float * 512)(), np.zeros(512, np.float32), 1.0):
            for call in (lambda: be.quant_matvec_into(w, bad, 0, y), lambda: be.quant_matvec_into(w, x, bad, y),
                         lambda: be.quant_matvec_into(w, x, 0, y, 1, bad),
                         lambda: be.quant_matmul_into(w, bad, 1, "bf16", 0, 0, y), lambda: be.quant_matmul_into(w, x, 1, "bf16", bad, 0, y)):
                try:
                    call()
                except TypeError:
                    refused += 1
        n = len(launches())
        be.quant_matvec_into(w, np.int64(x), 0, np.uint64(y))
        be.quant_matvec_into(w, x, None, y, 1, None)
        result = refused, n
    """)
    assert refused == 25 and launched == 0
