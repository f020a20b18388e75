"""Measured workloads of the engine: what programs have it do, through its public entry points.

Four kinds of work, over the sizes, types and options that programs use:

- ``spi``: one token through the tensor SPI as a host program drives it (gather an embedding row, quantMatvec,
  quantMatvecAdd, an output head, download, release): every result is a buffer of its own, and latency counts.
- ``matvec``: ``quant_matvec_into``, one projection in each of ``layers`` layers, weights of every layer distinct
  (a decode step reads each weight once), batch 1 and up, optionally onto a residual.
- ``decode``: a captured decode step (``decode_plan``), all projections of ``layers`` decoder layers and a head.
- ``matmul``: ``quant_matmul_into``, the prefill product, one projection in each of ``layers`` layers.

Weights are GGUF blocks of normally distributed values, made on the GPU from the seed. ``exact`` decodes the same blocks
with plain torch in 64 bits.
"""
from __future__ import annotations

import torch

from jax4j_amd import Mi355xBackend, QuantType

_BE = Mi355xBackend()
_DEV = "cuda:0"


def listed():
    return [
        # one token of a small model through the SPI: a handful of calls, each a few microseconds of GPU work
        dict(name="spi_token_q4_0_d1024", kind="spi", type="Q4_0", d=1024, vocab=4096),
        # attention-output-sized projection, one request
        dict(name="matvec_q8_0_4096x4096_b1", kind="matvec", type="Q8_0", rows=4096, cols=4096, batch=1, layers=16, add=True),
        # low-bit weights of a shape that divides by nothing in particular
        dict(name="matvec_q2_0_8189x3200_b1", kind="matvec", type="Q2_0", rows=8189, cols=3200, batch=1, layers=16, add=False),
        # a few requests decoded together
        dict(name="matvec_q4_0_11008x4096_b5", kind="matvec", type="Q4_0", rows=11008, cols=4096, batch=5, layers=8, add=False),
        # many requests decoded together, the wide projection back to the model width
        dict(name="matvec_q6_k_4096x14336_b61", kind="matvec", type="Q6_K", rows=4096, cols=14336, batch=61, layers=4, add=True),
        # the decode step of the benchmark (Llama-3-8B shapes, Q4_K_M mix), one request and sixteen
        dict(name="decode_q4_k_m_b1", kind="decode", mix="Q4_K_M", d=4096, kv=1024, ffn=14336, vocab=128256, layers=32, batch=1),
        dict(name="decode_q4_k_m_b16", kind="decode", mix="Q4_K_M", d=4096, kv=1024, ffn=14336, vocab=128256, layers=32, batch=16),
        # prefill of a prompt of 512 tokens on quantized activations
        dict(name="matmul_q8_0_int8_m512", kind="matmul", type="Q8_0", variant="int8", m=512, rows=4096, cols=4096, layers=4),
        # ... and of 2048 tokens with bf16 activations
        dict(name="matmul_q8_0_bf16_m2048", kind="matmul", type="Q8_0", variant="bf16", m=2048, rows=4096, cols=4096, layers=4),
        # a short prompt (or one chunk of a chat turn)
        dict(name="matmul_q4_k_bf16_m24", kind="matmul", type="Q4_K", variant="bf16", m=24, rows=14336, cols=4096, layers=4),
        # the largest projection of a prefill
        dict(name="matmul_q4_k_bf16_m2048", kind="matmul", type="Q4_K", variant="bf16", m=2048, rows=14336, cols=4096, layers=2),
        # a prompt of no round length
        dict(name="matmul_q6_k_bf16_m777", kind="matmul", type="Q6_K", variant="bf16", m=777, rows=4096, cols=14336, layers=2),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _cols(rng, lo, hi, unit):
    return max(unit, _log(rng, lo, hi) // unit * unit)


def draw(rng):
    kind = rng.choice(["spi", "matvec", "matvec", "decode", "matmul", "matmul", "matmul"])
    if kind == "spi":
        t = rng.choice(["Q8_0", "Q4_0", "Q4_K", "Q6_K", "Q2_0"])
        return dict(kind=kind, type=t, d=_cols(rng, 512, 4096, 256), vocab=_log(rng, 512, 32000))
    if kind == "matvec":
        t = rng.choice(["Q8_0", "Q4_0", "Q4_K", "Q6_K", "Q2_0"])
        unit = getattr(QuantType, t).block_elements
        batch = rng.choice([1, 1, _log(rng, 2, 64)])
        if t == "Q2_0":
            batch = min(batch, 8)
        return dict(kind=kind, type=t, rows=_log(rng, 512, 32768), cols=_cols(rng, 512, 14336, unit), batch=batch,
                    layers=rng.choice([2, 4, 8]), add=rng.random() < 0.5)
    if kind == "decode":
        return dict(kind=kind, mix=rng.choice(["Q4_K_M", "Q4_K_M", "Q8_0", "Q4_0"]), d=_cols(rng, 1024, 4096, 256),
                    kv=_cols(rng, 256, 1024, 64), ffn=_cols(rng, 2048, 14336, 256), vocab=_log(rng, 4000, 64000),
                    layers=rng.randint(2, 8), batch=_log(rng, 1, 32))
    t = rng.choice(["Q8_0", "Q8_0", "Q4_0", "Q4_K", "Q6_K"])
    variant = rng.choice(["int8", "bf16"]) if t == "Q8_0" else "bf16"
    return dict(kind=kind, type=t, variant=variant, m=_log(rng, 8, 2048), rows=_log(rng, 512, 14336),
                cols=_cols(rng, 1024, 8192, 32 if t == "Q8_0" else 256), layers=2)


# ---- inputs ----------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(seed)


def _normal_codes(g, shape, spread, zero, lo, hi):
    return (torch.randn(shape, generator=g, device=_DEV) * spread + zero).round_().clamp_(lo, hi)


def _scales(g, n, mean):
    """fp16 block scales of about `mean`, as two bytes each."""
    s = torch.rand((n, 1), generator=g, device=_DEV).mul_(0.8 * mean).add_(0.6 * mean)
    return s.to(torch.float16).view(torch.uint8)


def _blocks(g, qtype, rows, cols):
    """GGUF blocks [blocks, block bytes] (uint8) of a [rows, cols] matrix of about N(0, 0.02) weights."""
    n = rows * cols // qtype.block_elements
    if qtype is QuantType.Q8_0:
        q = _normal_codes(g, (n, 32), 42.0, 0.0, -127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_scales(g, n, 0.02 / 42), q], 1)
    if qtype is QuantType.Q4_0:
        q = _normal_codes(g, (n, 32), 2.7, 8.0, 0, 15).to(torch.uint8)
        return torch.cat([_scales(g, n, 0.02 / 2.7), q[:, :16] | (q[:, 16:] << 4)], 1)
    if qtype is QuantType.Q2_0:
        q = torch.randint(0, 4, (n, 32, 4), generator=g, device=_DEV, dtype=torch.uint8)
        return torch.cat([_scales(g, n, 0.016), q[..., 0] | (q[..., 1] << 2) | (q[..., 2] << 4) | (q[..., 3] << 6)], 1)
    if qtype is QuantType.Q4_K:
        q = _normal_codes(g, (n, 4, 2, 32), 2.7, 7.5, 0, 15).to(torch.uint8)
        sc = torch.randint(24, 64, (n, 8), generator=g, device=_DEV, dtype=torch.uint8)
        # the mins of a block of about zero mean: the scales, with dmin 7.5 times d
        packed = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), sc[:, :4] | ((sc[:, 4:] >> 4) << 6),
                            (sc[:, 4:] & 15) | ((sc[:, 4:] & 15) << 4)], 1)
        d = torch.rand((n, 1), generator=g, device=_DEV).mul_(0.8).add_(0.6) * (0.02 / (2.7 * 44))
        dd = torch.cat([d, 7.5 * d], 1).to(torch.float16).view(torch.uint8)
        return torch.cat([dd, packed, (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(n, 128)], 1)
    if qtype is QuantType.Q6_K:
        q = _normal_codes(g, (n, 2, 4, 32), 10.0, 32.0, 0, 63).to(torch.uint8)
        ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
        qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        sc = torch.randint(40, 128, (n, 16), generator=g, device=_DEV) * (
            2 * torch.randint(0, 2, (n, 16), generator=g, device=_DEV) - 1)
        return torch.cat([ql.reshape(n, 128), qh.reshape(n, 64), sc.to(torch.int8).view(torch.uint8),
                          _scales(g, n, 0.02 / (10 * 84))], 1)
    raise ValueError(qtype)


def _decode64(qtype, b, rows, cols):
    """The fp64 values of GGUF blocks."""
    def half(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double()

    n = b.shape[0]
    if qtype is QuantType.Q8_0:
        w = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif qtype is QuantType.Q4_0:
        w = half(0) * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8)
    elif qtype is QuantType.Q2_0:
        w = half(0) * (torch.stack([(b[:, 2:] >> s) & 3 for s in (0, 2, 4, 6)], 2).reshape(n, 128).double() - 1)
    elif qtype is QuantType.Q4_K:
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32).double()
        w = (half(0) * sc)[..., None] * q - (half(2) * mn)[..., None]
    else:
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 32)
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
        q = q.reshape(n, 16, 16).double() - 32
        w = (half(208) * b[:, 192:208].contiguous().view(torch.int8).double())[..., None] * q
    return w.reshape(rows, cols)


def _activations(g, *shape):
    """Activations of a normalised layer: N(0, 1), and a few channels an order of magnitude larger."""
    x = torch.randn(shape, generator=g, device=_DEV)
    big = torch.rand(shape[-1:], generator=g, device=_DEV) < 0.002
    return torch.where(big, 8 * x, x)


_PROJECTIONS = ("q", "k", "v", "o", "gate", "up", "down")


def _decode_shapes(case):
    """{projection: (type, rows, cols)} of a layer, and of the head."""
    d, kv, ffn = case["d"], case["kv"], case["ffn"]
    wide = QuantType.Q4_K if case["mix"] == "Q4_K_M" else getattr(QuantType, case["mix"])
    fine = QuantType.Q6_K if case["mix"] == "Q4_K_M" else wide
    return {"q": (wide, d, d), "k": (wide, kv, d), "v": (wide, kv, d), "o": (wide, d, d), "gate": (wide, ffn, d),
            "up": (wide, ffn, d), "down": (fine, d, ffn), "head": (wide, case["vocab"], d)}


def _weight_shapes(case):
    """(type, rows, cols) of every matrix of the case, in the order in which its blocks are made."""
    if case["kind"] == "spi":
        t = getattr(QuantType, case["type"])
        return [(t, case["vocab"], case["d"]), (t, case["d"], case["d"]), (t, case["d"], case["d"])]
    if case["kind"] == "decode":
        s = _decode_shapes(case)
        return [s[p] for _ in range(case["layers"]) for p in _PROJECTIONS] + [s["head"]]
    return [(getattr(QuantType, case["type"]), case["rows"], case["cols"])] * case["layers"]


def _dense_inputs(case, g):
    """The activations, from a generator of their own."""
    kind = case["kind"]
    if kind == "spi":
        return {"token": int(torch.randint(0, case["vocab"], (1,), generator=g, device=_DEV))}
    if kind == "matvec":
        n, b = case["layers"], case["batch"]
        return {"x": [_activations(g, b, case["cols"]) for _ in range(n)],
                "add": [torch.randn((b, case["rows"]), generator=g, device=_DEV) for _ in range(n)] if case["add"] else None}
    if kind == "decode":
        b = case["batch"]
        return {"h0": _activations(g, b, case["d"]), "x_o": _activations(g, b, case["d"]), "x_down": _activations(g, b, case["ffn"])}
    return {"x": [_activations(g, case["m"], case["cols"]).to(torch.bfloat16) for _ in range(case["layers"])]}


class _State:
    """What a program holds between calls; gives its engine buffers back when it goes."""

    def __init__(self):
        self.weights, self.plan = [], None

    def __del__(self):
        torch.cuda.synchronize()
        if self.plan is not None:
            self.plan.destroy()
        for w in self.weights:
            _BE.release(w)


def prepare(case, seed):
    s = _State()
    s.case = case
    gw = _gen(2 * seed)
    for qtype, rows, cols in _weight_shapes(case):
        b = _blocks(gw, qtype, rows, cols)
        torch.cuda.synchronize()  # the upload reads the blocks on the engine's stream
        s.weights.append(_BE.upload_quantized_device(b.data_ptr(), b.numel(), qtype, (rows, cols)))
    for k, v in _dense_inputs(case, _gen(2 * seed + 1)).items():
        setattr(s, k, v)
    f32 = dict(device=_DEV, dtype=torch.float32)
    if case["kind"] == "matvec":
        s.y = [torch.empty((case["batch"], case["rows"]), **f32) for _ in s.weights]
    elif case["kind"] == "matmul":
        s.y = [torch.empty((case["m"], case["rows"]), **f32) for _ in s.weights]
        int8 = case["variant"] == "int8"
        s.xq = torch.empty((case["m"], case["cols"]), device=_DEV, dtype=torch.int8) if int8 else None
        s.xs = torch.empty((case["m"], case["cols"] // 32), **f32) if int8 else None
    elif case["kind"] == "decode":
        n, b = case["layers"], case["batch"]
        s.h = s.h0.clone()
        s.qkv = torch.empty((n, b, case["d"] + 2 * case["kv"]), **f32)
        s.gate_up = torch.empty((n, b, 2 * case["ffn"]), **f32)
        s.logits = torch.empty((b, case["vocab"]), **f32)
        per = len(_PROJECTIONS)
        layers = [dict(zip(_PROJECTIONS, s.weights[per * i:per * i + per])) for i in range(n)]
        io = {k: getattr(s, k).data_ptr() for k in ("h", "x_o", "x_down", "qkv", "gate_up", "logits")}
        s.plan = _BE.decode_plan(layers, s.weights[-1], b, io)
        s.stream = torch.cuda.ExternalStream(_BE.stream())
    torch.cuda.synchronize()
    return s


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "matvec":
        for i, w in enumerate(s.weights):
            _BE.quant_matvec_into(w, s.x[i].data_ptr(), s.add[i].data_ptr() if case["add"] else 0, s.y[i].data_ptr(), case["batch"])
        return s.y
    if kind == "matmul":
        xq, xs = (s.xq.data_ptr(), s.xs.data_ptr()) if case["variant"] == "int8" else (0, 0)
        for i, w in enumerate(s.weights):
            _BE.quant_matmul_into(w, s.x[i].data_ptr(), case["m"], case["variant"], xq, xs, s.y[i].data_ptr())
        return s.y
    if kind == "decode":
        with torch.cuda.stream(s.stream):  # the next token's embeddings
            s.h.copy_(s.h0)
        s.plan.run()
        return {"h": s.h, "qkv": s.qkv, "gate_up": s.gate_up, "logits": s.logits}
    emb, up, out = s.weights
    x = _BE.quant_gather_row(emb, s.token)
    u = _BE.quant_matvec(up, x)
    y = _BE.quant_matvec_add(out, u, x)
    logits = _BE.quant_matvec(emb, y)
    got = {"y": _BE.download(y), "logits": _BE.download(logits)}
    for b in (x, u, y, logits):
        _BE.release(b)
    return got


def _weight_bytes(case):
    return sum(t.byte_size_for(rows * cols) for t, rows, cols in _weight_shapes(case))


def work(case):
    kind = case["kind"]
    elements = sum(rows * cols for _, rows, cols in _weight_shapes(case))
    if kind == "spi":  # the head's matrix also holds the embedding row
        return {"bytes": _weight_bytes(case) + 4 * (4 * case["d"] + case["vocab"]), "flops": 2 * elements}
    if kind == "matvec":
        n, b = case["layers"], case["batch"]
        dense = 4 * n * b * (case["cols"] + case["rows"] * (2 if case["add"] else 1))
        return {"bytes": _weight_bytes(case) + dense, "flops": 2 * elements * b}
    if kind == "decode":
        b, n = case["batch"], case["layers"]
        dense = 4 * b * (n * (case["d"] + 2 * case["kv"] + 2 * case["ffn"]) + 4 * case["d"] + case["ffn"] + case["vocab"])
        return {"bytes": _weight_bytes(case) + dense, "flops": 2 * elements * b}
    n, m = case["layers"], case["m"]
    return {"bytes": _weight_bytes(case) + n * m * (2 * case["cols"] + 4 * case["rows"]), "flops": 2 * elements * m}


def tolerance(case):
    if case["kind"] == "matmul" and case["variant"] == "bf16":
        return {"rel": 7e-3}  # weights rounded to bf16: 1.7e-3 from the 64-bit product
    if case["kind"] in ("matvec", "decode") and case["batch"] >= 3:
        return {"rel": 2e-4}  # block sums rounded inside the matrix cores: 5e-5 from the 64-bit product
    return {"rel": 4e-6}  # 32-bit sums of exact products (int8: of the same quantized activations): up to 6e-7


def _quantized64(x):
    """bf16 activations as the int8 variant sees them: per 32, fp32 scale amax / 127, round half away."""
    b = x.float().reshape(*x.shape[:-1], -1, 32)
    s = b.abs().amax(-1, keepdim=True)
    s = s / torch.full_like(s, 127.0)  # a tensor: division by a number multiplies by its reciprocal
    v = b * torch.where(s != 0, 1.0 / s, torch.zeros_like(s))
    q = (torch.sign(v) * torch.floor(v.abs() + 0.5)).clamp(-127, 127)
    return (q.double() * s.double()).reshape(x.shape)


def exact(case, seed):
    kind, gw = case["kind"], _gen(2 * seed)
    d = _dense_inputs(case, _gen(2 * seed + 1))

    def weights():
        for qtype, rows, cols in _weight_shapes(case):
            yield _decode64(qtype, _blocks(gw, qtype, rows, cols), rows, cols)

    if kind == "matvec":
        y = [x.double() @ w.t() for x, w in zip(d["x"], weights())]
        return [a + b.double() for a, b in zip(y, d["add"])] if case["add"] else y
    if kind == "matmul":
        return [(_quantized64(x) if case["variant"] == "int8" else x.double()) @ w.t() for x, w in zip(d["x"], weights())]
    if kind == "spi":
        emb, up, out = weights()
        x = emb[d["token"]]
        y = out @ (up @ x) + x
        return {"y": y.cpu().numpy(), "logits": (emb @ y).cpu().numpy()}
    h, x_o, x_down = d["h0"].double(), d["x_o"].double(), d["x_down"].double()
    it, qkv, gate_up = weights(), [], []
    for _ in range(case["layers"]):
        qkv.append(torch.cat([h @ next(it).t() for _ in range(3)], 1))
        h = x_o @ next(it).t() + h
        gate_up.append(torch.cat([h @ next(it).t() for _ in range(2)], 1))
        h = x_down @ next(it).t() + h
    return {"h": h, "qkv": torch.stack(qkv), "gate_up": torch.stack(gate_up), "logits": h @ next(it).t()}
