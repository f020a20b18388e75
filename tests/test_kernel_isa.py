"""Properties of the built kernels' machine code that their source relies on and no result shows for sure.

The tile kernels (gemm_tile.h, gemv_tile.h) load X for all waves of a workgroup and W for the loading
wave alone, and at every second stage wait for all but the newest unit of W before the barrier. A
load of X issued behind one of W would still be in flight when other waves read it."""
from __future__ import annotations

import re
import struct
import subprocess

import pytest

from jax4j_amd import _native as N

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14


def code_objects():
    """The gfx950 code objects in the library's offload bundles."""
    data = N.LIB_PATH.read_bytes()
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen].decode()
            p += 24 + idlen
            if "gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 24)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: its LDS loads (the resource registers), waits and barriers, in order}"""
    folder, found = tmp_path_factory.mktemp("isa"), {}
    for i, obj in enumerate(code_objects()):
        path = folder / f"{i}.co"
        path.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], capture_output=True, text=True, check=True).stdout
        name = None
        for line in text.splitlines():
            if m := re.match(r"<(\S+)>:", line):
                name = m[1] if "_tileILi" in m[1] else None
                if name:
                    found[name] = []
            elif name:
                if m := re.search(r"buffer_load_dword\S* v\d+, (s\[\d+:\d+\]).* lds", line):
                    found[name].append(m[1])
                elif m := re.search(r"s_waitcnt .*vmcnt\((\d+)\)", line):
                    found[name].append(int(m[1]))
                elif "s_barrier" in line:
                    found[name].append("barrier")
    return found


def test_tile_kernels_issue_x_before_w(kernels):
    assert len(kernels) >= 30 and any("gemv_tile" in k for k in kernels)
    for name, seq in kernels.items():
        if m := re.search(r"gemm_tileILi(\d+)ELi(\d+)ELi(\d+)E", name):
            fmt, waves, tm = map(int, m.groups())
            x_loads = 4 * tm // waves
        else:
            fmt, tm = map(int, re.search(r"gemv_tileILi(\d+)ELi(\d+)E", name).groups())
            x_loads = 2 * tm + (tm if fmt == Q4_K else 0)
        w_loads = (4 if fmt == Q8_0 else 2) + (3 if fmt == Q6_K else 1)
        # prologue: a unit of W, the first stage of X, another unit of W
        first = [v for v in seq[:seq.index("barrier")] if isinstance(v, str)]
        x = set(first[w_loads:w_loads + x_loads])
        assert len(first) == 2 * w_loads + x_loads and not x & {*first[:w_loads], *first[w_loads + x_loads:]}, name
        behind = w_loads  # loads of W that may be outstanding at the barrier
        waited, stages = None, 0
        segment = []
        for v in seq:
            if isinstance(v, int):
                waited = v if waited is None else min(waited, v)
            elif v != "barrier":
                waited = None
                segment.append(v)
            else:
                if stages:
                    kinds = "".join("x" if r in x else "w" for r in segment)
                    assert kinds in ("", "x" * x_loads, "x" * x_loads + "w" * w_loads), (name, stages, kinds)
                    if segment:
                        behind = kinds.count("w")
                if segment:
                    assert waited is not None and waited <= behind, (name, stages, waited)
                stages, segment, waited = stages + 1, [], None
        assert stages >= 4, name
