"""GPU parity of the LDS-tiled bf16 prefill GEMM (tiles of 32, 64, 96, 128, 160 rows x 128 columns on
four waves, 128 and 256 rows x 256 on eight, K split over workgroups or not) against the CPU
oracle, through the C ABI.

Bar: within 2e-5 * ||y||inf of the fp64 product of X and the bf16-rounded weights (only the fp32
accumulation order differs), repeated calls bit for bit, and one-hot rows of X give bf16 of a
weight column bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from jax4j_amd import DType, QuantType
from jax4j_amd import synthetic as S

pytestmark = pytest.mark.gpu

TOL_ACCUM = 2e-5
ALL = [QuantType.Q8_0, QuantType.Q4_0, QuantType.Q4_K, QuantType.Q6_K]


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


# Rows and columns past the last tile, one superblock up to many, K splits of unequal length. Q8_0 also
# with an odd number of 64-element stages (K = 192).
SHAPES = [(5, 37, 512), (24, 4096, 4096), (70, 130, 1280), (97, 10007, 256), (90, 5001, 3072), (160, 14336, 512),
          (777, 4097, 768), (1024, 4096, 256), (300, 14336, 256), (2049, 14337, 256), (512, 14336, 512), (2048, 14336, 256),
          (950, 1040, 2560), (500, 1041, 1280), (700, 700, 1024)]


# Every tile at a depth where its loop comes round several times, over an odd number of superblocks (so that
# Q6_K's d changes its half of a dword within a row): (row tiles of 32, waves, K groups) (1, 4, 1), (2, 4, 1),
# (3, 4, 1), (4, 4, 1), (5, 4, 1), (4, 8, 1), (8, 8, 1); for the types with K groups (1, 2, 2), (2, 2, 2),
# (1, 2, 4), (2, 2, 4), (3, 2, 4), (2, 4, 2); and K splits. test_gemm_tile_choice.py checks that they are picked.
DEEP = [(130, 6001, 1280), (350, 4097, 1280), (500, 4097, 1280), (500, 6001, 1280), (2049, 2049, 1280), (1025, 6001, 1280), (2049, 6001, 1280),
        (33, 129, 1280), (500, 1041, 1280), (200, 2049, 1792), (300, 2047, 3840), (600, 2001, 2304), (523, 3459, 1792),
        (30, 1205, 3840), (140, 1205, 4352), (257, 2049, 4352)]


@pytest.mark.parametrize("qt", ALL, ids=lambda q: q.name)
@pytest.mark.parametrize("m,n,k", SHAPES + [(12, 20000, 192), (2048, 2049, 64)] + DEEP)
def test_gemm_tiles_match_oracle(backend, qt, m, n, k):
    if k % 256 and qt is not QuantType.Q8_0:
        pytest.skip("K of a whole number of superblocks")
    print("[case] gemm tile", qt.name, m, n, k, flush=True)
    seed = 9000 + m + n + k
    w_blob = S.quant_blocks(qt, seed, n, k)
    xb = S.activations_bf16(seed + 1, m * k).reshape(m, k)
    w = backend.upload_quantized(w_blob, qt, (n, k))
    x = backend.upload(xb, shape=(m, k), dtype=DType.BF16)
    y = backend.quant_matmul(w, x, "bf16")
    got = backend.download(y).reshape(m, n)
    rows = sorted({0, 1, 31, 32, m // 2, m - 2, m - 1} & set(range(m)))
    ref = oracle.gemm_f64(np.ascontiguousarray(xb[rows]), w_blob, len(rows), n, k, bf16_weights=True, qtype=qt.id)
    assert np.isfinite(got).all()
    assert np.abs(got[rows] - ref).max() <= TOL_ACCUM * np.abs(ref).max()
    y2 = backend.quant_matmul(w, x, "bf16")
    assert np.array_equal(bits(backend.download(y2)), bits(got).reshape(-1))
    for h in (w, x, y, y2):
        backend.release(h)


@pytest.mark.parametrize("qt", ALL, ids=lambda q: q.name)
def test_gemm_tile_one_hot_rows_return_bf16_weights(backend, qt):
    """Row r of X is e_{k_r}: row r of Y is bf16 of weight column k_r. The k_r cover every element of
    a 32-block in both blocks and both stages of a load unit, and both ends of K."""
    n, k = 20000, 512
    ks = sorted(set(list(range(0, 64)) + list(range(96, 128)) + [64, 80, 255, 256, 300, 383, 384, 511]))
    m = len(ks)
    w_blob = S.quant_blocks(qt, 93, n, k)
    xb = np.zeros((m, k), np.uint16)
    xb[np.arange(m), ks] = 0x3F80  # bf16 1.0
    w = backend.upload_quantized(w_blob, qt, (n, k))
    x = backend.upload(xb, shape=(m, k), dtype=DType.BF16)
    y = backend.quant_matmul(w, x, "bf16")
    got = backend.download(y).reshape(m, n)
    u = bits(oracle.dequant_matrix(qt.id, w_blob, n, k)[:, ks].T).astype(np.uint64)
    want = (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32).view(np.float32)
    assert np.array_equal(bits(got), bits(np.where(want == 0, np.float32(0.0), want)))
    for h in (w, x, y):
        backend.release(h)


@pytest.mark.parametrize("qt", ALL, ids=lambda q: q.name)
def test_gemm_tile_keeps_rows_apart(backend, qt):
    """Infinities and NaN in some rows of X reach those rows of Y alone."""
    m, n, k = 200, 700, 1024
    w_blob = S.quant_blocks(qt, 95, n, k)
    xb = S.activations_bf16(96, m * k).reshape(m, k)
    w = backend.upload_quantized(w_blob, qt, (n, k))
    x = backend.upload(xb, shape=(m, k), dtype=DType.BF16)
    clean = backend.quant_matmul(w, x, "bf16")
    bad = xb.copy()
    bad[7, 1000] = 0x7F80  # +inf
    bad[130, 3] = 0x7FC0  # NaN
    xbad = backend.upload(bad, shape=(m, k), dtype=DType.BF16)
    y = backend.quant_matmul(w, xbad, "bf16")
    got, ref = (backend.download(h).reshape(m, n) for h in (y, clean))
    keep = np.setdiff1d(np.arange(m), [7, 130])
    assert np.array_equal(bits(got[keep]), bits(ref[keep]))
    assert not np.isfinite(got[7]).any() and np.isnan(got[130]).all()
    for h in (w, x, clean, xbad, y):
        backend.release(h)
