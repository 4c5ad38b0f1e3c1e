"""What this framework is timed on: quantized linear layers and embedding lookups through its public entry points.

A case is a list of weights that meet one batch of activation rows ("linear": one qmatmul or int8 linear per weight, as
a layer of a model calls them), or a table whose rows are looked up ("rows"). Weights are loaded once, as a program
loads them: GGUF blocks through ops.prepare (16-row tiles for the types with kernel planes, the file's blocks for the
exact path's types), int8 per-channel weights through int8.repack. Activations are bfloat16, as the forward's are.

The listed cases are one 27B-class layer with its stacked projections (q|k|v, o, gate|up, down: synth.LAYER_27B_STACKED)
at the batch sizes an engine runs it (one row, the row buckets 4 and 16, a batch of 64, a prefill chunk of 512, a long
prefill of 2048), its smallest projections alone, a vocabulary head, a smaller model's ragged batch, the exact path in
decode and prefill, and the embedding lookup of a prefill chunk.
"""
import math

import torch

from mashbox_amd import int8, ops

BF16 = torch.bfloat16

# name -> (ggml type id, values per block, bytes per block, byte offsets of the block's fp16 scales)
BLOCKS = {
    "Q4_0": (2, 32, 18, (0,)), "Q8_0": (8, 32, 34, (0,)), "Q4_K": (12, 256, 144, (0, 2)),
    "Q5_K": (13, 256, 176, (0, 2)), "Q6_K": (14, 256, 210, (208,)),
    "Q4_1": (3, 32, 20, (0, 2)), "Q5_0": (6, 32, 22, (0,)), "Q5_1": (7, 32, 24, (0, 2)),
    "Q2_K": (10, 256, 84, (80, 82)), "Q3_K": (11, 256, 110, (108,)), "IQ4_NL": (20, 32, 18, (0,)),
    "IQ4_XS": (23, 256, 136, (0,)), "F16": (1, 1, 2, ()), "BF16": (30, 1, 2, ()),
}
PLANES = ("Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K", "int8")                # the types with kernel planes
EXACT = ("Q4_1", "Q5_0", "Q5_1", "Q2_K", "Q3_K", "IQ4_NL", "IQ4_XS", "F16", "BF16")     # the exact path's


def listed():
    def linear(name, rows, weights):
        return {"name": name, "kind": "linear", "rows": rows, "weights": weights}

    def layer(t):
        return "%s 8192x5120, %s 5120x6144, %s 34816x5120, %s 5120x17408" % (t, t, t, t)

    return [
        # the smallest calls of a decode step: two key/value projections of one token
        linear("kv_q4k_1", 1, "Q4_K 1024x5120, Q4_K 1024x5120"),
        # decode of one sequence: every layer of every token runs this
        linear("layer_q4k_1", 1, layer("Q4_K")),
        # decode of four sequences on a mixed file (v and down in six bits, the rest in four, as _M files have it)
        linear("layer_q4k_q6k_4", 4, "Q4_K 7168x5120, Q6_K 1024x5120, Q4_K 5120x6144, Q4_K 34816x5120, Q6_K 5120x17408"),
        # decode of sixteen sequences on eight-bit blocks
        linear("layer_q8_16", 16, layer("Q8_0")),
        # continuous batching: 64 tokens on int8 per-channel weights
        linear("layer_int8_64", 64, layer("int8")),
        # a ragged batch on a smaller model's odd sizes (rows, outputs and a K that no tile divides)
        linear("ragged_q5k_37", 37, "Q5_K 3083x2816, Q5_K 2816x2816, Q5_K 15001x2816, Q5_K 2816x7680"),
        # one chunk of a chunked prefill
        linear("chunk_q4k_512", 512, layer("Q4_K")),
        # a long prompt's prefill, the largest batch the engine cuts
        linear("prefill_q4k_2048", 2048, layer("Q4_K")),
        # the vocabulary head of one decoded token
        linear("head_q6k_1", 1, "Q6_K 151936x2560"),
        # the exact path in decode: a three-bit file's layer, one token
        linear("layer_q3k_1", 1, layer("Q3_K")),
        # the exact path in prefill: a chunk on a code-book four-bit file's layer
        linear("chunk_iq4xs_512", 512, layer("IQ4_XS")),
        # the embedding lookup of a prefill chunk
        {"name": "embed_q6k_512", "kind": "rows", "rows": 512, "weights": "Q6_K 151936x2560"},
    ]


def _spread(rng, lo, hi, step=1):
    """a multiple of step in [lo, hi], spread over the logarithm"""
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + step))) // step * step)))


def draw(rng):
    kind = rng.choice(("planes", "planes", "planes", "exact", "exact", "rows"))
    t = rng.choice(EXACT if kind == "exact" else PLANES)
    step = 16 if t == "int8" else max(32, BLOCKS[t][1])
    if kind == "rows":
        k = _spread(rng, 512, 8192, step)
        return {"kind": "rows", "rows": _spread(rng, 1, 2048), "weights": "%s %dx%d" % (t, _spread(rng, 1000, 151936 * 2560 // max(k, 2560)), k)}
    m = _spread(rng, 1, 512 if kind == "exact" else 2048)
    weights = []
    for _ in range(rng.choice((1, 2, 3))):
        k = _spread(rng, 512, 17408, step)
        n = _spread(rng, 256, min(34816, 34816 * 5120 // k // 2))
        if kind == "exact" and n * k > ops.EXACT_CHUNK:    # large ones of whole 16-row groups, as files have them
            n = n // 16 * 16
        weights.append("%s %dx%d" % (t, n, k))
    return {"kind": "linear", "rows": m, "weights": ", ".join(weights)}


def _weights(case):
    out = []
    for part in case["weights"].split(","):
        t, size = part.split()
        n, k = (int(v) for v in size.split("x"))
        out.append((t, n, k))
    return out


def _raw(gen, t, n, k):
    """a weight of seeded random codes as the file holds it, block scales ~ U(1e-3, 1e-2) (int8: q, s); the float types
    ~ N(0, 0.05)"""
    def scales(shape):
        return torch.rand(shape, generator=gen, device="cuda") * 9e-3 + 1e-3

    if t == "int8":
        return torch.randint(-127, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8), scales((n,))
    _, values, size, at = BLOCKS[t]
    if values == 1:
        w = torch.randn((n, k), generator=gen, device="cuda") * 0.05
        return w.to(torch.float16 if t == "F16" else BF16).view(torch.uint8).reshape(n, -1)
    raw = torch.randint(0, 256, (n * (k // values), size), generator=gen, device="cuda", dtype=torch.uint8)
    for o in at:
        raw[:, o:o + 2] = scales((raw.shape[0], 1)).to(torch.float16).view(torch.uint8)
    return raw.reshape(n, -1)


def _inputs(case, seed):
    """per weight its type, sizes and blocks, and the activations (one batch per row length) or the looked-up ids"""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    weights = _weights(case)
    if case["kind"] == "rows":
        ins = torch.randint(0, weights[0][1], (case["rows"],), generator=gen, device="cuda", dtype=torch.int32)
    else:
        ins = {}
        for _, _, k in weights:
            if k not in ins:
                ins[k] = torch.randn((case["rows"], k), generator=gen, device="cuda").to(BF16)
    for t, n, k in weights:
        yield t, n, k, _raw(gen, t, n, k), ins if case["kind"] == "rows" else ins[k]


def prepare(case, seed):
    if not ops.kernel_types():
        ops.load_kernels()
    state = []
    for t, n, k, raw, x in _inputs(case, seed):
        if t == "int8" and case["kind"] == "rows":
            w = {"q": raw[0], "s": raw[1]}
        elif t == "int8":
            w = int8.repack(*raw)
        else:
            w = ops.prepare(raw, BLOCKS[t][0], (n, k))
        state.append((case["kind"], t, w, x))
    return state


def run(state):
    out = []
    for kind, t, w, x in state:
        if kind == "rows":
            out.append(int8.embed(w, x) if t == "int8" else ops.take_rows(w, x))
        else:
            out.append(int8.linear(x, w) if t == "int8" else ops.qmatmul(x, w))
    return out


def work(case):
    m, nbytes, flops = case["rows"], 0, 0
    for t, n, k in _weights(case):
        per_row = k + 4 if t == "int8" else k // BLOCKS[t][1] * BLOCKS[t][2]
        if case["kind"] == "rows":                      # the looked-up rows and the ids read, float32 (int8: bf16) written
            nbytes += m * (per_row + 4 + (2 if t == "int8" else 4) * k)
            flops += m * k
        else:
            nbytes += n * per_row + 2 * m * n
            flops += 2 * m * n * k
    if case["kind"] != "rows":
        nbytes += sum(2 * m * k for k in {k for _, _, k in _weights(case)})
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # a lookup is exact. A product's error against 64 bits is its rounding to bfloat16 (relative 2-norm 1.7e-3), and
    # where the batched kernels round the weight to bfloat16 too, 2.4e-3; about four times that
    if case["kind"] == "rows":
        return "exact"
    return {"rel": 7e-3 if case["weights"].split()[0] in EXACT else 1e-2, "max": 5e-2}


# ------------------------------------------------------------------------------------- the same in 64 bits, plain torch
IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _f16(b, o):
    return b[:, o:o + 2].contiguous().view(torch.float16).double()


def _nibbles(q):
    return torch.cat([q & 15, q >> 4], -1)


def _scale_min(b):
    """Q4_K / Q5_K: the 8 six-bit scales and mins of 12 bytes"""
    lo, mid, hi = b[:, 4:8], b[:, 8:12], b[:, 12:16]
    return torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1).double(), torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1).double()


def _dequant(t, raw, k):
    """(rows, row_bytes) blocks -> float64 (rows, k)"""
    n = raw.shape[0]
    if t in ("F16", "BF16"):
        return raw.contiguous().view(torch.float16 if t == "F16" else BF16).double()
    b = raw.reshape(-1, BLOCKS[t][2])
    if t == "Q4_0":
        w = _f16(b, 0) * (_nibbles(b[:, 2:]).double() - 8)
    elif t == "Q8_0":
        w = _f16(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif t == "Q4_1":
        w = _f16(b, 0) * _nibbles(b[:, 4:]).double() + _f16(b, 2)
    elif t in ("Q5_0", "Q5_1"):
        o = 2 if t == "Q5_0" else 4
        bit = torch.stack([(b[:, o + i // 8] >> (i % 8)) & 1 for i in range(32)], 1)
        q = (_nibbles(b[:, o + 4:]) | (bit << 4)).double()
        w = _f16(b, 0) * (q - 16) if t == "Q5_0" else _f16(b, 0) * q + _f16(b, 2)
    elif t in ("IQ4_NL", "IQ4_XS"):
        book = torch.tensor(IQ4, dtype=torch.float64, device=raw.device)
        if t == "IQ4_NL":
            w = _f16(b, 0) * book[_nibbles(b[:, 2:]).long()]
        else:
            lo = torch.stack([b[:, 4:8] & 15, b[:, 4:8] >> 4], -1).reshape(-1, 8)
            hi = torch.stack([(b[:, 2 + j // 4] >> (2 * (j % 4))) & 3 for j in range(8)], 1)
            s = (lo | (hi << 4)).double() - 32
            w = (_f16(b, 0) * s)[:, :, None] * book[_nibbles(b[:, 8:].reshape(-1, 8, 16)).long()]
    elif t in ("Q4_K", "Q5_K"):
        s, m = _scale_min(b)
        q = b[:, -128:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        if t == "Q5_K":
            q = q | (torch.stack([(b[:, 16:48] >> j) & 1 for j in range(8)], 1) << 4)
        w = (_f16(b, 0) * s)[:, :, None] * q.double() - (_f16(b, 2) * m)[:, :, None]
    elif t == "Q6_K":
        lo = b[:, :128].reshape(-1, 2, 1, 64)
        lo = torch.cat([lo & 15, lo >> 4], 2).reshape(-1, 2, 4, 32)
        hi = torch.stack([(b[:, 128:192].reshape(-1, 2, 32) >> (2 * r)) & 3 for r in range(4)], 2)
        s = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (_f16(b, 208) * s)[:, :, None] * ((lo | (hi << 4)).double() - 32).reshape(-1, 16, 16)
    elif t == "Q2_K":
        q = torch.stack([(b[:, 16:80].reshape(-1, 2, 32) >> (2 * j)) & 3 for j in range(4)], 2).reshape(-1, 16, 16).double()
        w = (_f16(b, 80) * (b[:, :16] & 15).double())[:, :, None] * q - (_f16(b, 82) * (b[:, :16] >> 4).double())[:, :, None]
    else:                                                # Q3_K
        lo = torch.cat([b[:, 96:104] & 15, b[:, 96:104] >> 4], 1)
        hi = torch.cat([(b[:, 104:108] >> (2 * j)) & 3 for j in range(4)], 1)
        s = (lo | (hi << 4)).double() - 32
        q = torch.stack([(b[:, 32:96].reshape(-1, 2, 32) >> (2 * j)) & 3 for j in range(4)], 2).reshape(-1, 8, 32)
        h = torch.stack([(b[:, :32] >> j) & 1 for j in range(8)], 1)
        w = (_f16(b, 108) * s)[:, :, None] * (q.double() - 4 * (1 - h.double())).reshape(-1, 16, 16)
    return w.reshape(n, k)


def exact(case, seed):
    out = []
    for t, n, k, raw, x in _inputs(case, seed):
        if case["kind"] == "rows":
            i = x.long()
            out.append(raw[0][i].double() * raw[1][i].double()[:, None] if t == "int8" else _dequant(t, raw[i], k))
            continue
        xd, parts = x.double(), []
        for r in range(0, n, 4096):
            w = raw[0][r:r + 4096].double() * raw[1][r:r + 4096].double()[:, None] if t == "int8" else _dequant(t, raw[r:r + 4096], k)
            parts.append(torch.matmul(xd, w.t().contiguous()))
        out.append(torch.cat(parts, 1))
    return out
