"""Decode plans of 9 to 16 rows, where the window sums of a GEMV ride on the next launch: equal bit for
bit to the same step as single engine calls, in every case in which they ride, go to their place in a
group of several types, or must not wait (the next launch too small, rows not a multiple of 4, buffers of
the caller that overlap)."""
from __future__ import annotations

import numpy as np
import pytest

from jax4j_amd import QuantType
from jax4j_amd import synthetic as S

pytestmark = pytest.mark.gpu

Q4, Q6, Q8 = QuantType.Q4_K, QuantType.Q6_K, QuantType.Q8_0
NAMES = ("q", "k", "v", "o", "gate", "up", "down")
# (types, rows of q, k, v, ffn): one type (a launch per group), two types in a group with the sums placed
# by the next launch, with a next launch of one tile, and with row counts that float4 sums cannot take
CASES = {
    "one type": ((Q4,) * 7, 512, 64, 64, 2304),
    "placed": ((Q4, Q4, Q6, Q4, Q8, Q4, Q6), 2048, 64, 128, 2304),
    "small next launch": ((Q4, Q4, Q6, Q4, Q4, Q4, Q4), 4096, 64, 16, 2304),
    "odd rows": ((Q4, Q4, Q6, Q4, Q4, Q4, Q4), 510, 63, 65, 2304),
}
D = 4352  # three column windows of 16 rows


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


@pytest.mark.parametrize("case,b", [("one type", 9), ("one type", 16), ("placed", 12), ("placed", 16),
                                    ("small next launch", 16), ("odd rows", 13)])
@pytest.mark.parametrize("overlap", [False, True])
def test_plan_window_sums(backend, case, b, overlap):
    print("[case] plan sums", case, b, overlap, flush=True)
    types, qr, kr, vr, ffn = CASES[case]
    rows = dict(q=qr, k=kr, v=vr, o=D, gate=ffn, up=ffn, down=D)
    cols = dict(q=D, k=D, v=D, o=2048, gate=D, up=D, down=ffn)
    w = {n: backend.upload_quantized(S.quant_blocks(t, 300 + i, rows[n], cols[n]), t, (rows[n], cols[n]))
         for i, (n, t) in enumerate(zip(NAMES, types))}
    L, qkv = 2, qr + kr + vr
    h0 = S.activations_f32(1, b * D)
    nq, ng = L * b * qkv, L * b * 2 * ffn
    buf = {n: backend.upload(v) for n, v in dict(h=h0, xo=S.activations_f32(2, b * 2048), xd=S.activations_f32(3, b * ffn),
                                                 qkv=np.zeros(max(nq, b * 2048), np.float32), gu=np.zeros(ng, np.float32)).items()}
    ptr = {n: backend.buffer_desc(x).device_ptr for n, x in buf.items()}
    if overlap:  # o reads what q|k|v of layer 0 wrote, down what gate|up of layer 0 wrote
        ptr["xo"], ptr["xd"] = ptr["qkv"], ptr["gu"]
    io = dict(h=ptr["h"], x_o=ptr["xo"], x_down=ptr["xd"], qkv=ptr["qkv"], gate_up=ptr["gu"], logits=0)
    plan = backend.decode_plan([w] * L, None, b, io)
    try:
        plan.run()
        backend.sync()
        got = [backend.download(buf[n]) for n in ("h", "qkv", "gu")]
    finally:
        plan.destroy()

    def mv(n, x, add=None):
        bx = backend.upload(x, shape=x.shape)
        if add is None:
            by = backend.quant_matvec(w[n], bx)
        else:
            ba = backend.upload(add, shape=add.shape)
            by = backend.quant_matvec_add(w[n], bx, ba)
            backend.release(ba)
        out = backend.download(by).reshape(b, -1)
        backend.release(bx)
        backend.release(by)
        return out

    h, qs, gs = h0.reshape(b, D), np.zeros(max(nq, b * 2048), np.float32), np.zeros(ng, np.float32)
    xo, xd = S.activations_f32(2, b * 2048), S.activations_f32(3, b * ffn)
    for l in range(L):
        qs[l * b * qkv:(l + 1) * b * qkv] = np.concatenate([mv(n, h) for n in "qkv"], axis=1).reshape(-1)
        h = mv("o", (qs[:b * 2048] if overlap else xo).reshape(b, 2048), h)
        gs[l * b * 2 * ffn:(l + 1) * b * 2 * ffn] = np.concatenate([mv(n, h) for n in ("gate", "up")], axis=1).reshape(-1)
        h = mv("down", (gs[:b * ffn] if overlap else xd).reshape(b, ffn), h)
    for name, g, e in zip(("h", "qkv", "gate_up"), got, (h.reshape(-1), qs, gs)):
        assert np.array_equal(bits(g), bits(e)), name
    for x in (*w.values(), *buf.values()):
        backend.release(x)
