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
