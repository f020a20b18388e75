"""GPU parity of the tiled batched GEMV (more rows of x than the 16-row kernel takes in a launch or
two: from 19 rows for Q8_0 and Q6_K, 27 or 35 for Q4_K and Q4_0) against the CPU oracle.

Bar, relative to a row's ||y||inf: 1e-5, where x contributes 2^-22 by its two fp16 parts and each of
the K / 32 block sums and folds 2^-23 of its size, which random signs keep near sqrt(K / 32) of
them; Q4_K 4e-5, the bound of the 16-row kernel, since its min term cancels most of what the codes
sum up to.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from jax4j_amd import QuantType
from jax4j_amd import synthetic as S

pytestmark = pytest.mark.gpu

ALL = [QuantType.Q8_0, QuantType.Q4_0, QuantType.Q4_K, QuantType.Q6_K]


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def matvec(backend, w, xs):
    x = backend.upload(xs, shape=xs.shape)
    y = backend.quant_matvec(w, x)
    out = backend.download(y).reshape(xs.shape[0], -1)
    backend.release(x)
    backend.release(y)
    return out


# Rows of x at the first of each rule, full and ragged tiles of 32 and (the last two, and 65 x 20001)
# of 64, and past a chunk of 256;
# rows of W around a tile of 128; K of one split (512), of unequal splits (768: 512 + 256; 5120: 5 of
# 1024; 2816: 768 three times and 512), of many splits (9216, 33024).
SHAPES = [(19, 129, 512), (27, 127, 5120), (32, 300, 768), (33, 1, 2816), (35, 257, 2048), (64, 128, 512),
          (65, 130, 768), (257, 70, 512), (35, 40, 9216), (36, 33, 33024), (257, 12500, 512), (130, 5001, 2816)]
# All K splits in one workgroup: tiles of 32 and of 64 rows, three splits and two, the last one shorter.
ALL_SPLITS = [(65, 9001, 1280), (250, 15001, 768)]


@pytest.mark.parametrize("qt", ALL, ids=lambda q: q.name)
@pytest.mark.parametrize("b,n,k", SHAPES + ALL_SPLITS + [(19, 65, 64), (20, 140, 576), (40, 129, 1088), (70, 20, 640), (65, 20001, 576),
                                                       (65, 9001, 1344), (66, 9001, 1408)])
def test_gemv_tiles_match_oracle(backend, qt, b, n, k):
    if k % (64 if qt is QuantType.Q8_0 else 128 if qt is QuantType.Q4_0 else 256):
        pytest.skip("K of a whole number of blocks of the split layout")
    print("[case] gemv tile", qt.name, b, n, k, flush=True)
    blob = S.quant_blocks(qt, 7000 + b + n + k, n, k)
    w = backend.upload_quantized(blob, qt, (n, k))
    xs = S.activations_f32(b + n + k, b * k).reshape(b, k) * np.exp2(np.arange(b) % 40 - 20.0).astype(np.float32)[:, None]
    xs[1] = 0
    add = S.activations_f32(b + n, b * n).reshape(b, n)
    got = matvec(backend, w, xs)
    ref = oracle.matmul_f64(qt.id, blob, n, k, xs)
    bar = 4e-5 if qt is QuantType.Q4_K else 1e-5
    # one row of W: no row maximum to measure against, but the sum of its terms' sizes
    size = np.abs(ref).max(axis=1) if n > 1 else np.abs(xs.astype(np.float64)) @ np.abs(oracle.dequant_matrix(qt.id, blob, n, k)[0].astype(np.float64))
    assert (np.abs(got - ref).max(axis=1) <= bar * size).all()
    assert not bits(got[1] + np.float32(0)).any()
    # a row does not depend on the other rows, and an infinite one stays by itself
    xs2 = xs.copy()
    xs2[2, 3] = np.inf
    got2 = matvec(backend, w, xs2)
    assert np.array_equal(bits(np.delete(got2, 2, 0)), bits(np.delete(got, 2, 0)))
    assert not np.isfinite(got2[2]).any()
    # add joins last, also where it is y
    x, res = backend.upload(xs, shape=(b, k)), backend.upload(add.reshape(-1))
    rp = backend.buffer_desc(res).device_ptr
    backend.quant_matvec_into(w, backend.buffer_desc(x).device_ptr, rp, rp, b)
    backend.sync()
    assert np.array_equal(bits(backend.download(res).reshape(b, n)), bits(got + add))
    for h in (w, x, res):
        backend.release(h)


@pytest.mark.parametrize("qt", ALL, ids=lambda q: q.name)
def test_gemv_tile_sums_do_not_depend_on_the_launch(backend, qt):
    """The K splits depend on the columns alone: rows of x in a larger batch, and rows of W in a
    larger matrix, give the same bits; single products come out of the codes exactly."""
    k = 2816
    blobs = [S.quant_blocks(qt, 81 + i, n, k) for i, n in enumerate((100, 1500))]
    ws = [backend.upload_quantized(b, qt, (n, k)) for b, n in zip(blobs, (100, 1500))]
    both = backend.concat_rows(ws)
    xs = S.activations_f32(5, 300 * k).reshape(300, k)
    y0, y1 = (matvec(backend, w, xs[:35]) for w in ws)
    assert np.array_equal(bits(matvec(backend, both, xs)[:35]), bits(np.concatenate([y0, y1], axis=1)))
    # one-hot rows of a power of two: what the code, scale and min of one element give, to fp32 rounding
    ks = np.r_[0:64, 255, 256, 300, 511, 512, 1023, 1024, 2815]
    hot = np.zeros((len(ks), k), np.float32)
    hot[np.arange(len(ks)), ks] = 4.0
    want = 4.0 * oracle.dequant_matrix(qt.id, blobs[0], 100, k)[:, ks].T.astype(np.float64)
    got = matvec(backend, ws[0], hot)
    if qt is QuantType.Q4_K:  # two rounded terms, each up to 16 times the result's block
        assert np.abs(got - want).max() <= 2.0**-20 * np.abs(want).max()
    else:
        assert np.abs(got - want).max() <= 2.0**-23 * np.abs(want).max()
    for h in (*ws, both):
        backend.release(h)


@pytest.mark.parametrize("qt", ALL, ids=lambda q: q.name)
@pytest.mark.parametrize("b,n,k", ALL_SPLITS)
def test_gemv_tile_sums_do_not_depend_on_where_the_splits_run(backend, qt, b, n, k):
    """Rows of W in a matrix so large that a workgroup runs every split give the bits that they give
    alone, with a workgroup per split."""
    blobs = [S.quant_blocks(qt, 91 + i, r, k) for i, r in enumerate((100, n - 100))]
    ws = [backend.upload_quantized(blob, qt, (r, k)) for blob, r in zip(blobs, (100, n - 100))]
    both = backend.concat_rows(ws)
    xs = S.activations_f32(6, b * k).reshape(b, k)
    xs[3] = 0
    assert np.array_equal(bits(matvec(backend, both, xs)[:, :100]), bits(matvec(backend, ws[0], xs)))
    for h in (*ws, both):
        backend.release(h)


# (bytes of a block, offset of its scales, their bytes)
SCALES = {QuantType.Q8_0: (34, 0, 2), QuantType.Q4_0: (18, 0, 2), QuantType.Q4_K: (144, 0, 4), QuantType.Q6_K: (210, 208, 2)}


@pytest.mark.parametrize("qt", ALL, ids=lambda q: q.name)
@pytest.mark.parametrize("large", [3.0e5, 3.0e12])
def test_a_large_element_of_x_costs_other_splits_no_bits(backend, qt, large):
    """x is scaled per K split (2816 columns: 768 three times and 512). Where the weights of the first split are
    zero, an element of x there changes nothing. Where they are zero in its block alone, the others of
    its split keep an absolute error of 2^-35 of it, and of 2^-22 of themselves."""
    b, n, k = 40, 200, 2816
    bb, at, nb = SCALES[qt]
    x = S.activations_f32(3, b * k).reshape(b, k)
    x[:, 5] = 0
    xl = x.copy()
    xl[:, 5] = large
    for cols in (768, qt.block_elements):
        blocks = S.quant_blocks(qt, 77, n, k).reshape(n, k // qt.block_elements, bb).copy()
        blocks[:, :cols // qt.block_elements, at:at + nb] = 0
        w = backend.upload_quantized(blocks.reshape(-1), qt, (n, k))
        got, plain = matvec(backend, w, xl), matvec(backend, w, x)
        if cols == 768:
            assert np.array_equal(bits(got), bits(plain))
        wf = np.abs(oracle.dequant_matrix(qt.id, blocks.reshape(-1), n, k).astype(np.float64))
        ref = oracle.matmul_f64(qt.id, blocks.reshape(-1), n, k, xl)
        # Q4_K's products of codes and of mins are each up to 16 times their difference
        size = (16 if qt is QuantType.Q4_K else 1) * (2.0**-22 * (np.abs(x).astype(np.float64) @ wf.T) + 2.0**-35 * large * wf[:, :768].sum(axis=1))
        bar = 4e-5 if qt is QuantType.Q4_K else 1e-5
        assert (np.abs(got - ref) <= bar * np.abs(ref).max(axis=1, keepdims=True) + size).all()
        backend.release(w)
