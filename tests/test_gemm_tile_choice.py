"""Which instances of the tile kernels the sizes of the GPU tests run, by the launch model in the library (on
a HIP runtime that logs launches, fakehip.py). A change of the model that leaves an instance without
a test at depth fails here."""
from __future__ import annotations

import re

import fakehip
from test_gpu_gemm_tile import DEEP
from test_gpu_gemv_tile import ALL_SPLITS, SHAPES as GEMV_SHAPES

FORMATS = {2: "Q4_0", 8: "Q8_0", 12: "Q4_K", 14: "Q6_K"}


def instance(kernel, name):
    m = re.search(name + r"I((?:L[ib]\d+E)+)E", kernel)
    return m and tuple(map(int, re.findall(r"L[ib](\d+)E", m[1])))


def picked(shim, call, sizes, name):
    """{format: instances}, and the instances in the library."""
    kernels, calls = fakehip.run(shim, f"""
        result = [], []
        result[0][:] = fake.fake_kernels().decode().split()
        for t in {list(FORMATS.values())}:
            qt = getattr(QuantType, t)
            for m, n, k in {sizes!r}:
                w = zeros(qt, n, k)
                log()
                assert lib.{call} == 0, N.last_error()
                result[1].append([t, m, n, k, [l[1:5] for l in launches()]])
                be.release(w)
    """)
    library = {i for k in kernels if (i := instance(k, name))}
    return library, [(t, m, n, k, i, l[3]) for t, m, n, k, ls in calls for l in ls if (i := instance(l[0], name))]


def test_every_gemm_tile_is_tested_at_depth(tmp_path):
    library, runs = picked(fakehip.build_shim(tmp_path), "j4q_quant_matmul_into(w.handle, 4096, m, 1, None, None, 4096, None)", DEEP, "gemm_tile")
    assert len(library) == 7 + 3 * 13
    assert all(k // 256 % 2 and k >= 1280 for _, _, k in DEEP)
    assert library == {i for *_, i, splits in runs if splits == "1"}
    for f in (2, 12, 14):  # K splits over several tiles
        assert len({i for *_, i, splits in runs if int(splits) > 1 and i[0] == f}) >= 2


def test_every_gemv_tile_is_tested(tmp_path):
    library, runs = picked(fakehip.build_shim(tmp_path), "j4q_quant_matvec_into(w.handle, 4096, None, 4096, m, None)",
                           GEMV_SHAPES + ALL_SPLITS, "gemv_tile")
    one, several = ({i for *_, i, splits in runs if (int(splits) > 1) == s} for s in (False, True))
    assert len(library) == 16  # (format, row tiles of 32, whether a workgroup runs every split)
    assert library == one and {i for i in library if not i[2]} == several
