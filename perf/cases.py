"""The calls a user of this package makes, as measurable cases.

The shapes are those of the repository's own configurations: a 27B-class
dense layer (hidden 5120, 48 query and 8 KV heads of 128, FFN 17408,
vocabulary 151936) and a 4096 x 4096 projection, in the GGUF encodings such
files mix (Q4_K with Q6_K for the value, down and output matrices; Q8_0, Q5_K
and IQ4_XS files). The operations are the engine's: the decode matvec, merged
segments, one whole decode step, speculative verification of a few tokens, and
prompts of tens to thousands of tokens.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) weights in HBM, activations and output buffers
    run(state)          one pass through nuclis_amd.Backend / nuclis_amd.layer
    work(case)          bytes and flops the pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   what run returns, in float64 torch
"""
from __future__ import annotations

import numpy as np
import torch

import nuclis_amd as nq
from nuclis_amd import layer as nl

ENCODINGS = {"q8_0": nq.Q8_0, "q4_k": nq.Q4_K, "q5_k": nq.Q5_K, "q6_k": nq.Q6_K, "iq4_xs": nq.IQ4_XS}


def listed():
    return [
        # The smallest product of a decode step: the value projection of one
        # token, which mixed Q4_K files store as Q6_K. Latency and launches.
        {"name": "decode_v_q6_k", "op": "matvec", "enc": "q6_k", "rows": 1024, "columns": 5120},
        # A small square projection of an 8-bit file.
        {"name": "decode_q8_0_4096", "op": "matvec", "enc": "q8_0", "rows": 4096, "columns": 4096},
        # The gate (or up) matrix of one token: the bandwidth-bound decode product.
        {"name": "decode_gate_q4_k", "op": "matvec", "enc": "q4_k", "rows": 17408, "columns": 5120},
        # gate and up merged, with the SiLU epilogue, of a 4-bit non-linear file.
        {"name": "decode_pair_iq4_xs", "op": "pair", "enc": "iq4_xs", "rows": 17408, "columns": 5120},
        # One whole decode step: every projection of the layer and the output head.
        {"name": "decode_layer", "op": "layer", "vocab": nl.VOCAB},
        # Verification of two drafted tokens: F32 activations as the engine holds them.
        {"name": "verify3_down_q4_k", "op": "matmul", "enc": "q4_k", "rows": 5120, "columns": 17408, "tokens": 3, "x": "f32"},
        # Verification of seven drafted tokens, f16 activations.
        {"name": "verify8_gate_q4_k", "op": "matmul", "enc": "q4_k", "rows": 17408, "columns": 5120, "tokens": 8, "x": "f16"},
        # The same pass through the 6-bit down matrix of a mixed file, F32 activations.
        {"name": "verify8_down_q6_k", "op": "matmul", "enc": "q6_k", "rows": 5120, "columns": 17408, "tokens": 8, "x": "f32"},
        # A short chat turn through the attention output matrix: tens of tokens, a ragged count.
        {"name": "prompt77_o_q5_k", "op": "matmul", "enc": "q5_k", "rows": 5120, "columns": 6144, "tokens": 77, "x": "f32"},
        # One prompt chunk of 512 tokens.
        {"name": "prefill512_gate_q4_k", "op": "matmul", "enc": "q4_k", "rows": 17408, "columns": 5120, "tokens": 512, "x": "f16"},
        # A long prompt of a ragged length through the 6-bit down matrix, F32 activations.
        {"name": "prefill1999_down_q6_k", "op": "matmul", "enc": "q6_k", "rows": 5120, "columns": 17408, "tokens": 1999, "x": "f32"},
        # The largest: a 4096-token prompt chunk through the gate matrix.
        {"name": "prefill4096_gate_q4_k", "op": "matmul", "enc": "q4_k", "rows": 17408, "columns": 5120, "tokens": 4096, "x": "f16"},
    ]


def _log(rng, low, high):
    return low * (high / low) ** rng.random()


def draw(rng):
    """Matvecs of any row count and whole blocks per row, pairs of 16-row
    multiples, products of 2..4096 tokens with 8-row multiples, and layers of
    other vocabularies."""
    op = rng.choice(["matvec", "matvec", "pair", "matmul", "matmul", "matmul", "matmul", "matmul", "layer"])
    if op == "layer":
        return {"op": "layer", "vocab": int(_log(rng, 32000, nl.VOCAB)) // 16 * 16}
    enc = rng.choice(sorted(ENCODINGS))
    columns = max(4, int(_log(rng, 2048, 17408) / 256)) * 256
    rows = int(_log(rng, 1024, 20480))
    if op == "matvec":
        if enc == "q8_0" and rng.random() < 0.3:
            columns += 32 * rng.randrange(1, 8)
        return {"op": op, "enc": enc, "rows": rows, "columns": columns}
    if op == "pair":
        return {"op": op, "enc": enc, "rows": rows // 16 * 16, "columns": columns}
    tokens = int(_log(rng, 2, 4096))
    rows = rows // 8 * 8
    while tokens > 2 and rows * columns * tokens > 17408 * 5120 * 4096:
        tokens //= 2
    return {"op": op, "enc": enc, "rows": rows, "columns": columns, "tokens": tokens,
            "x": rng.choice(["f16", "f32"])}


# -- inputs -------------------------------------------------------------------

_backend = None


def backend():
    global _backend
    if _backend is None:
        _backend = nq.Backend(0)
    return _backend


POOL_ROWS, POOL_COLUMNS = 64, 8192


def weights(enc, rows, columns, seed, g):
    """[rows][row bytes] of GGUF blocks on the GPU: blocks drawn with
    repetition from a pool of N(0, 0.02) weights that the package's quantizer
    encoded, so codes and scales are distributed as in a file."""
    values, size = nq.LAYOUT[enc]
    w = np.random.default_rng(seed).standard_normal((POOL_ROWS, POOL_COLUMNS), dtype=np.float32)
    w *= np.float32(0.02)
    pool = torch.from_numpy(nq.quantize(enc, w)).cuda().view(-1, size)
    per_row = columns // values
    out = torch.empty((rows, per_row * size), dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 22) // per_row)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        pick = torch.randint(pool.shape[0], (n * per_row,), device="cuda", generator=g)
        out[r:r + n] = pool[pick].view(n, per_row * size)
    return out


def activations(shape, g):
    """N(0, 1) with channels of different strength, as hidden states have."""
    x = torch.randn(shape, device="cuda", generator=g)
    return x * torch.exp(0.5 * torch.randn(shape[-1], device="cuda", generator=g))


def matrix(enc, rows, columns, seed, g):
    return nq.Matrix(enc, rows, columns, weights(enc, rows, columns, seed, g))


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = {"op": case["op"], "backend": backend()}
    if case["op"] == "layer":
        shapes = dict(nl.SHAPES, lm_head=(nq.Q6_K, case["vocab"], nl.HIDDEN, 0))
        mats = {name: matrix(enc, rows, cols, seed + i, g)
                for i, (name, (enc, rows, cols, _)) in enumerate(shapes.items())}
        empty = lambda n: torch.empty(n, device="cuda")  # noqa: E731
        head = torch.arange(nl.Q_ROWS, device="cuda")
        bufs = {"qkv": empty(nl.Q_ROWS + 2 * nl.KV_ROWS), "h1": empty(nl.HIDDEN), "attn_o": empty(nl.HIDDEN),
                "act": empty(nl.FFN), "h2": empty(nl.HIDDEN), "down": empty(nl.HIDDEN), "logits": empty(case["vocab"]),
                "attn": empty(nl.Q_ROWS),
                "gqa_index": head // (nl.HEAD_DIM * nl.GQA) * nl.HEAD_DIM + head % nl.HEAD_DIM}
        s.update(layer=nl.DeviceLayer(mats, bufs), x=activations((nl.HIDDEN,), g))
        return s
    enc, rows, columns = ENCODINGS[case["enc"]], case["rows"], case["columns"]
    s["m"] = matrix(enc, rows, columns, seed, g)
    if case["op"] == "pair":
        s["up"] = matrix(enc, rows, columns, seed + 1, g)
    if case["op"] == "matmul":
        t = case["tokens"]
        x = activations((t, columns), g)
        s.update(x=x.half() if case["x"] == "f16" else x, y=torch.empty((t, rows), device="cuda"))
    else:
        s.update(x=activations((columns,), g), y=torch.empty(rows, device="cuda"))
    return s


def run(s):
    b = s["backend"]
    if s["op"] == "layer":
        nl.step(b, s["layer"], s["x"])
        return {"h2": s["layer"].buffers["h2"], "logits": s["layer"].buffers["logits"]}
    m, x, y = s["m"], s["x"], s["y"]
    if s["op"] == "matvec":
        b.matvec(m, x, y)
    elif s["op"] == "pair":
        b.matvec_segments([(m, y), (s["up"], y)], x, nq.SEGMENT_SILU_MUL_PAIR)
    else:
        b.matmul(m, x, m.columns, y, m.rows, x.shape[0])
    return y


# -- what a pass needs, and what it should give ----------------------------------


def work(case):
    if case["op"] == "layer":
        shapes = dict(nl.SHAPES, lm_head=(nq.Q6_K, case["vocab"], nl.HIDDEN, 0)).values()
        weight = sum(rows * nq.row_bytes(enc, cols) for enc, rows, cols, _ in shapes)
        return {"bytes": weight + 4 * (3 * nl.HIDDEN + case["vocab"]),
                "flops": sum(2 * rows * cols for _, rows, cols, _ in shapes)}
    rows, columns = case["rows"], case["columns"]
    mats = 2 if case["op"] == "pair" else 1
    tokens = case.get("tokens", 1)
    x_bytes = 2 if case.get("x") == "f16" else 4
    weight = mats * rows * nq.row_bytes(ENCODINGS[case["enc"]], columns)
    return {"bytes": weight + tokens * (columns * x_bytes + rows * 4), "flops": 2 * mats * tokens * rows * columns}


def tolerance(case):
    # Products of one token, and of up to three F32 tokens where the encoding
    # has a row kernel, hold F32 sums; the tiles round weights or activations
    # to f16.
    if case["op"] == "layer":
        return {"rel": 5e-6}
    if case["op"] in ("matvec", "pair") or (case["tokens"] <= 3 and case["x"] == "f32"
                                            and case["enc"] in ("q8_0", "q4_k", "q6_k")):
        return {"rel": 3e-6}
    return {"rel": 1.2e-3}


def _half(b, at):
    return b[..., at:at + 2].contiguous().view(torch.float16).double()


def _groups_k(b):
    """The eight 6-bit scales and minima of Q4_K / Q5_K blocks."""
    s = b[..., 4:16].int()
    scale = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | (s[..., 0:4] >> 6 << 4)], -1)
    minimum = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | (s[..., 4:8] >> 6 << 4)], -1)
    return (_half(b, 0) * scale).unsqueeze(-1), (_half(b, 2) * minimum).unsqueeze(-1)


def decode(enc, raw):
    """float64 values of GGUF blocks: [rows][row bytes] -> [rows][columns]."""
    values, size = nq.LAYOUT[enc]
    b = raw.view(raw.shape[0], -1, size)
    if enc == nq.Q8_0:
        v = _half(b, 0) * b[..., 2:].contiguous().view(torch.int8)
    elif enc in (nq.Q4_K, nq.Q5_K):
        q = b[..., -128:].view(*b.shape[:2], 4, 32)
        q = torch.stack([q & 15, q >> 4], -2).reshape(*b.shape[:2], 8, 32)
        if enc == nq.Q5_K:
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(8, 1)
            q = q | ((b[..., 16:48].unsqueeze(-2) >> bit & 1) << 4)
        scale, minimum = _groups_k(b)
        v = scale * q - minimum
    elif enc == nq.Q6_K:
        low = b[..., :128].view(*b.shape[:2], 2, 1, 2, 32)
        low = torch.cat([low & 15, low >> 4], -3).reshape(*b.shape[:2], 2, 4, 32)
        shift = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8).view(4, 1)
        high = b[..., 128:192].view(*b.shape[:2], 2, 1, 32) >> shift & 3
        q = (low | high << 4).double().view(*b.shape[:2], 16, 16) - 32
        v = q * (_half(b, 208) * b[..., 192:208].contiguous().view(torch.int8)).unsqueeze(-1)
    else:
        table = torch.tensor([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113],
                             device=b.device, dtype=torch.float64)
        g = torch.arange(8, device=b.device)
        low = b[..., 4:8].int().repeat_interleave(2, -1) >> (4 * (g % 2)) & 15
        high = (b[..., 2:3].int() | b[..., 3:4].int() << 8) >> (2 * g) & 3
        scale = _half(b, 0) * ((low | high << 4) - 32)
        q = b[..., 8:].view(*b.shape[:2], 8, 16)
        v = table[torch.cat([q & 15, q >> 4], -1).long()] * scale.unsqueeze(-1)
    return v.reshape(raw.shape[0], -1)


def _product(m, x):
    """x [tokens][columns] (float64) by the rows of m, a slab of rows at a time."""
    out = torch.empty((x.shape[0], m.rows), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // m.columns)
    for r in range(0, m.rows, step):
        out[:, r:r + step] = x @ decode(m.encoding, m.bytes[r:r + step]).t().contiguous()
    return out


def _silu(v):
    return v * torch.sigmoid(v)


def exact(case, seed):
    s = prepare(case, seed)
    x = s["x"].double()
    if case["op"] == "layer":
        m = s["layer"].mats
        p = lambda name, v: _product(m[name], v.unsqueeze(0))[0]  # noqa: E731
        h1 = x + p("o", p("v", x)[s["layer"].buffers["gqa_index"]])
        h2 = h1 + p("down", _silu(p("gate", h1)) * p("up", h1))
        return {"h2": h2, "logits": p("lm_head", h2)}
    if case["op"] == "matmul":
        return _product(s["m"], x)
    y = _product(s["m"], x.unsqueeze(0))[0]
    return _silu(y) * _product(s["up"], x.unsqueeze(0))[0] if case["op"] == "pair" else y
