"""Runs engine calls on the CPU: the built library, on a HIP runtime that allocates host memory and
launches nothing (fake_hip.cpp). What a call allocates, launches, waits for and refuses is then
visible without a GPU; results are not computed."""
from __future__ import annotations

import json
import subprocess
import sys
import textwrap
from pathlib import Path

TESTS = Path(__file__).resolve().parent
ROCM = Path("/opt/rocm")

_PRELUDE = """
import ctypes as C, json, sys
import numpy as np
fake = C.CDLL({shim!r}, mode=C.RTLD_GLOBAL)
fake.fake_log.restype = fake.fake_kernels.restype = C.c_char_p
fake.fake_used.restype = C.c_uint64
fake.fake_capacity.argtypes = [C.c_uint64]
fake.fake_capture.argtypes = [C.c_void_p, C.c_int]
sys.path.insert(0, {root!r})
from jax4j_amd import Mi355xBackend, QuantType, DType
from jax4j_amd import _native as N
be = Mi355xBackend()
lib = be._lib()
def log(*kinds):
    "The runtime calls since the last log(), of these kinds."
    lines = fake.fake_log().decode().split("\\n")[:-1]
    return [l for l in lines if not kinds or l.split()[0] in kinds]
def launches():
    return [l.split() for l in log("launch")]
def zeros(qt, rows, cols):
    return be.upload_quantized(np.zeros(qt.byte_size_for(rows * cols), np.uint8), qt, (rows, cols))
def address(n):
    "A 16-byte aligned address of n bytes of host memory, standing for the caller's device memory."
    a = np.zeros(n // 16 + 2, dtype=np.complex128)
    keep.append(a)
    return (a.ctypes.data + 15) // 16 * 16
keep = []
result = None
log()
"""


def build_shim(folder: Path) -> Path:
    """Compiles the runtime's stand-in into `folder`."""
    lib = folder / "fake_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM / 'include'}",
                    "-o", str(lib), str(TESTS / "fake_hip.cpp")], check=True)
    return lib


def run(shim_path: Path, body: str):
    """Runs `body` in a process of its own; returns what it assigns to `result`."""
    code = _PRELUDE.format(shim=str(shim_path), root=str(TESTS.parent)) + textwrap.dedent(body) + "\nprint('RESULT ' + json.dumps(result))\n"
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-4000:]
    return json.loads(p.stdout.split("RESULT ")[-1])
