"""The work that programs built on halo_amd spend their time in, as cases that can be timed and compared.

A model's forward pass over quantized weights is a sequence of these calls: the embedding rows and a norm, the token
mixers' projections, the FFN, the LM head; before it, the load of the weights. Each case runs one such piece through
halo_amd's public functions. Sizes are those of the hybrid layer with hidden size 5120 that bench.py times, and of the
4096 x 4096 Q4_0 matrix. A state holds several layers' weights where one layer is small, and a pass takes them in turn,
since a model's next layer never finds its weights in a cache.
"""
import math

import numpy as np
import torch

import halo_amd as hl

HIDDEN, HEADS, KV, INNER, GDN = 5120, 6144, 1024, 17408, 12288
EPS = 1e-6
COLD = 96 << 20  # bytes of weights that a decode state holds at least

# Weight types of one layer: gdn_in, gdn_out, q, k, v, o, gate and up, down
MIXES = {
    "q4_k_m": ("Q4_K", "Q4_K", "Q4_K", "Q4_K", "Q6_K", "Q4_K", "Q4_K", "Q6_K"),
    "ud": ("Q5_K", "Q5_K", "Q5_K", "IQ4_XS", "Q6_K", "Q5_K", "IQ4_XS", "Q5_K"),
}
BLOCK = {"F16": (1, 2), "Q4_0": (32, 18), "Q8_0": (32, 34), "Q3_K": (256, 110), "Q4_K": (256, 144), "Q5_K": (256, 176),
         "Q6_K": (256, 210), "IQ4_NL": (32, 18), "IQ4_XS": (256, 136)}
IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def row_bytes(t, cols):
    return cols // BLOCK[t][0] * BLOCK[t][1]


def layers_for(nbytes):
    return max(1, min(40, math.ceil(COLD / nbytes)))


def listed():
    return [
        # the smallest work: one projection at one token, called eagerly layer after layer; launch latency counts
        {"name": "proj_q4_0_4096_m1", "kind": "proj", "type": "Q4_0", "rows": 4096, "cols": 4096, "m": 1, "norm": False,
         "layers": 12, "graph": False},
        # a decode step of one layer, all projections with their fused norms, in a graph as a serving loop keeps it
        {"name": "layer_q4km_m1", "kind": "layer", "mix": "q4_k_m", "m": 1, "layers": 1, "graph": True},
        # the verify step of speculative decoding (two drafts and the last token) on a pack of Q5_K and IQ4_XS
        {"name": "layer_ud_m3", "kind": "layer", "mix": "ud", "m": 3, "layers": 1, "graph": True},
        # a few sequences or a short prompt: the FFN on a ragged handful of rows
        {"name": "ffn_iq4xs_m13", "kind": "ffn", "type": "IQ4_XS", "down": "Q5_K", "hidden": HIDDEN, "inner": INNER,
         "m": 13, "layers": 1, "graph": False},
        # a small prefill chunk
        {"name": "ffn_q4k_m64", "kind": "ffn", "type": "Q4_K", "down": "Q6_K", "hidden": HIDDEN, "inner": INNER, "m": 64,
         "layers": 1, "graph": False},
        # a full prefill chunk of the FFN: the largest part of a prompt's time
        {"name": "ffn_q4k_m512", "kind": "ffn", "type": "Q4_K", "down": "Q6_K", "hidden": HIDDEN, "inner": INNER, "m": 512,
         "layers": 1, "graph": False},
        # a prompt's ragged last chunk through the token mixers' projections (q, k and v in one grouped call)
        {"name": "mixer_q5k_m200", "kind": "mixer", "type": "Q5_K", "m": 200, "layers": 1, "graph": False},
        # the head over the whole vocabulary with its norm and argmax, one token
        {"name": "head_q6k_m1", "kind": "head", "type": "Q6_K", "rows": 248320, "valid": 248044, "cols": HIDDEN, "m": 1},
        # a prefill chunk's embedding rows and the first norm
        {"name": "embed_q6k_m512", "kind": "embed", "type": "Q6_K", "layout": "slab", "vocab": 151936, "cols": HIDDEN, "m": 512},
        # types without a SLAB form run on the file's own rows, in the CPU's order: a down projection at one token ...
        {"name": "gguf_iq4nl_m1", "kind": "gguf", "type": "IQ4_NL", "rows": HIDDEN, "cols": INNER, "m": 1, "layers": 2},
        # ... and a gate or up projection for a small prefill chunk
        {"name": "gguf_q3k_m64", "kind": "gguf", "type": "Q3_K", "rows": INNER, "cols": HIDDEN, "m": 64, "layers": 1},
        # load: the FFN weights of a layer from pageable host memory (as from a mapped file), gate and up row-fused
        {"name": "load_ffn", "kind": "load", "type": "Q5_K", "down": "Q6_K", "hidden": HIDDEN, "inner": INNER},
    ]


def log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("proj", "proj", "layer", "ffn", "ffn", "mixer", "head", "embed", "gguf", "load"))
    slab = ("Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K", "IQ4_XS")
    if kind == "proj":
        t = rng.choice(slab)
        rows, cols = log_int(rng, 500, INNER), 256 * log_int(rng, 8, 68)
        m = rng.choice((1, 1, 2, 3, 4, log_int(rng, 5, 512)))
        return {"kind": kind, "type": t, "rows": rows, "cols": cols, "m": m, "norm": rng.random() < 0.5,
                "layers": layers_for(rows * row_bytes(t, cols)) if m <= 8 else 1, "graph": rng.random() < 0.5}
    if kind == "layer":
        return {"kind": kind, "mix": rng.choice(sorted(MIXES)), "m": log_int(rng, 1, 8), "layers": 1, "graph": rng.random() < 0.7}
    if kind == "ffn":
        return {"kind": kind, "type": rng.choice(slab), "down": rng.choice(slab), "hidden": 256 * rng.randint(8, 20),
                "inner": 256 * rng.randint(24, 68), "m": log_int(rng, 1, 512), "layers": 1, "graph": rng.random() < 0.3}
    if kind == "mixer":
        return {"kind": kind, "type": rng.choice(("Q4_K", "Q5_K", "IQ4_XS")), "m": log_int(rng, 1, 512), "layers": 1,
                "graph": rng.random() < 0.3}
    if kind == "head":
        rows = log_int(rng, 32000, 248320)
        return {"kind": kind, "type": rng.choice(("Q6_K", "Q4_K", "Q5_K", "Q8_0")), "rows": rows, "valid": rows - rng.randint(0, 300),
                "cols": 256 * rng.randint(8, 20), "m": rng.choice((1, 1, 2, 3, 4))}
    if kind == "embed":
        t = rng.choice(("Q6_K", "Q4_K", "Q5_K", "Q8_0"))
        return {"kind": kind, "type": t, "layout": rng.choice(("slab", "gguf")), "vocab": log_int(rng, 32000, 151936),
                "cols": 256 * rng.randint(8, 20), "m": log_int(rng, 1, 512)}
    if kind == "gguf":
        t, m = rng.choice(("IQ4_NL", "Q3_K", "F16", "Q6_K")), log_int(rng, 1, 64)
        rows, cols = log_int(rng, 1000, 8000), 256 * log_int(rng, 8, 40)
        return {"kind": kind, "type": t, "rows": rows, "cols": cols, "m": m,
                "layers": layers_for(rows * row_bytes(t, cols)) if m == 1 else 1}
    return {"kind": kind, "type": rng.choice(slab), "down": rng.choice(slab), "hidden": 256 * rng.randint(8, 20),
            "inner": 256 * rng.randint(24, 60)}


# ---- weights: GGUF blocks with near-normal codes and scales that make W about N(0, 0.02) --------------------------


def generator(seed, *more):
    g = torch.Generator(device="cuda")
    k = seed
    for v in more:
        k = (k * 1000003 + v + 1) % (1 << 62)
    return g.manual_seed(k)


def normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def codes(g, shape, mid, sd, top):
    return normal(g, *shape).mul_(sd).add_(mid).round_().clamp_(0, top).to(torch.uint8)


def f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8)


def scale(g, shape, s):
    return f16_bytes(s * (1 + 0.15 * normal(g, *shape).clamp_(-3, 3)))


def nibbles(lo, hi):
    return lo | (hi << 4)


def k_scales(g, n):
    """The 12 bytes of 8 six-bit scales and mins (the mins near the scales, so that weights average to zero)."""
    sc = torch.randint(36, 64, (n, 8), generator=g, device="cuda")
    m = (sc + torch.randint(-2, 3, (n, 8), generator=g, device="cuda")).clamp_(0, 63)
    a = sc[:, :4] | (sc[:, 4:] >> 4 << 6)
    b = m[:, :4] | (m[:, 4:] >> 4 << 6)
    c = (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)
    return torch.cat([a, b, c], 1).to(torch.uint8)


def gguf(t, rows, cols, g):
    """rows x row_bytes of GGUF blocks on the GPU."""
    be, bb = BLOCK[t]
    n = rows * cols // be
    if t == "F16":
        return f16_bytes(0.02 * normal(g, rows, cols)).reshape(rows, -1)
    if t in ("Q4_0", "IQ4_NL"):
        q = codes(g, (n, 2, 16), 7.5, 3.0, 15)
        d = scale(g, (n, 1), 0.02 / 3.0 if t == "Q4_0" else 0.02 / 45.0)
        b = torch.cat([d, nibbles(q[:, 0], q[:, 1])], 1)
    elif t == "Q8_0":
        q = normal(g, n, 32).mul_(48).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        b = torch.cat([scale(g, (n, 1), 0.02 / 48.0), q], 1)
    elif t == "Q4_K":
        q = codes(g, (n, 4, 2, 32), 7.5, 3.2, 15)
        d = scale(g, (n, 1), 0.02 / 3.2 / 50)
        dm = f16_bytes(d.view(torch.float16) * 7.5)
        b = torch.cat([d, dm, k_scales(g, n), nibbles(q[:, :, 0], q[:, :, 1]).reshape(n, 128)], 1)
    elif t == "Q5_K":
        q = codes(g, (n, 4, 2, 32), 15.5, 6.5, 31)
        d = scale(g, (n, 1), 0.02 / 6.5 / 50)
        dm = f16_bytes(d.view(torch.float16) * 15.5)
        qh = torch.zeros((n, 32), dtype=torch.uint8, device="cuda")
        for j in range(8):
            qh |= (q[:, j // 2, j % 2] >> 4) << j
        b = torch.cat([d, dm, k_scales(g, n), qh, nibbles(q[:, :, 0] & 15, q[:, :, 1] & 15).reshape(n, 128)], 1)
    elif t == "Q6_K":
        q = codes(g, (n, 2, 4, 32), 32, 12, 63)  # element 128 n + 32 k + l
        ql = nibbles(q[:, :, :2] & 15, q[:, :, 2:] & 15).reshape(n, 128)
        qh = torch.zeros((n, 2, 32), dtype=torch.uint8, device="cuda")
        for k in range(4):
            qh |= (q[:, :, k] >> 4) << (2 * k)
        sc = torch.randint(70, 128, (n, 16), generator=g, device="cuda")
        sc = sc * (1 - 2 * torch.randint(0, 2, (n, 16), generator=g, device="cuda"))
        b = torch.cat([ql, qh.reshape(n, 64), sc.to(torch.int8).view(torch.uint8), scale(g, (n, 1), 0.02 / 12 / 100)], 1)
    elif t == "IQ4_XS":
        q = codes(g, (n, 8, 2, 16), 7.5, 3.0, 15)
        ls = torch.randint(4, 64, (n, 8), generator=g, device="cuda")
        sh = sum((ls[:, j] >> 4) << (2 * j) for j in range(8))
        sl = (ls[:, 0::2] & 15) | ((ls[:, 1::2] & 15) << 4)
        b = torch.cat([scale(g, (n, 1), 0.02 / 45 / 17), torch.stack([sh & 255, sh >> 8], 1).to(torch.uint8), sl.to(torch.uint8),
                       nibbles(q[:, :, 0], q[:, :, 1]).reshape(n, 128)], 1)
    else:  # Q3_K: element 128 n + 32 j + l
        q = codes(g, (n, 2, 4, 32), 4, 1.6, 7)
        qs = torch.zeros((n, 2, 32), dtype=torch.uint8, device="cuda")
        hm = torch.zeros((n, 32), dtype=torch.uint8, device="cuda")
        for i in range(2):
            for j in range(4):
                qs[:, i] |= (q[:, i, j] & 3) << (2 * j)
                hm |= (q[:, i, j] >> 2) << (4 * i + j)
        sc = torch.randint(4, 64, (n, 16), generator=g, device="cuda")
        lo = (sc[:, :8] & 15) | ((sc[:, 8:] & 15) << 4)
        hi = sum((sc[:, 4 * k:4 * k + 4] >> 4) << (2 * k) for k in range(4))
        b = torch.cat([hm, qs.reshape(n, 64), lo.to(torch.uint8), hi.to(torch.uint8), scale(g, (n, 1), 0.02 / 1.6 / 17)], 1)
    return b.reshape(rows, cols // be * bb)


def f64(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)


def dequant64(t, raw, cols):
    """The weights of GGUF rows in 64 bits, from the format's definition."""
    rows = raw.shape[0]
    be, bb = BLOCK[t]
    b = raw.reshape(-1, bb)
    n = b.shape[0]
    if t == "F16":
        return raw.contiguous().view(torch.float16).to(torch.float64)
    if t in ("Q4_0", "IQ4_NL"):
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).long()
        w = (q - 8).double() if t == "Q4_0" else torch.tensor(IQ4, device="cuda", dtype=torch.float64)[q]
        w = w * f64(b, 0)
    elif t == "Q8_0":
        w = b[:, 2:].contiguous().view(torch.int8).double() * f64(b, 0)
    elif t in ("Q4_K", "Q5_K"):
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1).double()
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
        p = b[:, bb - 128:].reshape(n, 4, 32)
        q = torch.stack([p & 15, p >> 4], 2).reshape(n, 8, 32)
        if t == "Q5_K":
            q = q | torch.stack([(b[:, 16:48] >> j & 1) << 4 for j in range(8)], 1)
        w = (f64(b, 0) * sc)[:, :, None] * q.double() - (f64(b, 2) * m)[:, :, None]
    elif t == "Q6_K":
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 32)
        q = torch.cat([ql & 15, ql >> 4], 2) | torch.stack([(qh >> (2 * k) & 3) << 4 for k in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * f64(b, 208)
        w = sc.reshape(n, 16, 1) * (q.double() - 32).reshape(n, 16, 16)
    elif t == "IQ4_XS":
        sh, sl = b[:, 2].int() | (b[:, 3].int() << 8), b[:, 4:8].int()
        ls = torch.stack([(sl[:, j // 2] >> (4 * (j % 2)) & 15) | ((sh >> (2 * j) & 3) << 4) for j in range(8)], 1)
        p = b[:, 8:].reshape(n, 8, 16)
        v = torch.tensor(IQ4, device="cuda", dtype=torch.float64)[torch.cat([p & 15, p >> 4], 2).long()]
        w = (f64(b, 0) * (ls - 32).double())[:, :, None] * v
    else:  # Q3_K
        s = b[:, 96:108].int()
        sc = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1) | torch.cat([(s[:, 8:] >> (2 * k) & 3) << 4 for k in range(4)], 1)
        qs = b[:, 32:96].reshape(n, 2, 32)
        q = torch.stack([torch.stack([(qs[:, i] >> (2 * j) & 3).double() - 4 * (1 - (b[:, :32] >> (4 * i + j) & 1).double())
                                      for j in range(4)], 1) for i in range(2)], 1)
        w = (f64(b, 108) * (sc - 32).double()).reshape(n, 16, 1) * q.reshape(n, 16, 16)
    return w.reshape(rows, cols)


# ---- the blocks of a forward pass, as steps over named tensors ----------------------------------------------------
# ("gemv" | "gate_up" | "group", [(type, rows, output), ...], cols, input, norm): the norm's weights are the input's own


def steps(case):
    k = case["kind"]
    if k == "proj":
        return [("gemv", [(case["type"], case["rows"], "y")], case["cols"], "x", case["norm"])]
    out = []
    if k in ("mixer", "layer"):
        t = MIXES[case["mix"]] if k == "layer" else (case["type"],) * 4 + ("Q6_K",) + (case["type"],) * 3
        out += [("gemv", [(t[0], GDN, "gdn_in")], HIDDEN, "x", True), ("gemv", [(t[1], HIDDEN, "gdn_out")], HEADS, "a", False),
                ("group", [(t[2], HEADS, "q"), (t[3], KV, "k"), (t[4], KV, "v")], HIDDEN, "x", True),
                ("gemv", [(t[5], HIDDEN, "o")], HEADS, "a", False)]
        if k == "mixer":
            return out
        gate, down, hidden, inner = t[6], t[7], HIDDEN, INNER
    else:
        gate, down, hidden, inner = case["type"], case["down"], case["hidden"], case["inner"]
    return out + [("gate_up", [(gate, inner, "act")], hidden, "x", True), ("gemv", [(down, hidden, "down")], inner, "act", False)]


def inputs(case, seed):
    """Activations and norm weights by name."""
    got = {}
    for i, (_, _, cols, name, norm) in enumerate(steps(case)):
        if name not in got and name != "act":
            got[name] = normal(generator(seed, 1, i), case["m"], cols)
            got[name + ".norm"] = 1 + 0.1 * normal(generator(seed, 2, i), cols)
    return got


def raw_weights(case, seed, layer):
    """Per step, the GGUF rows of its matrices (gate and up are two of one shape)."""
    for i, (op, mats, cols, _, _) in enumerate(steps(case)):
        yield [gguf(t, rows, cols, generator(seed, 3, layer, i, j)) for j, (t, rows, _) in enumerate(mats * (2 if op == "gate_up" else 1))]


def to_slab(t, raw, rows, cols):
    dst = torch.empty(hl.slab_bytes(hl.DType[t], rows, cols), dtype=torch.uint8, device="cuda")
    hl.repack_slab(hl.DType[t], raw, rows, cols, dst)
    return dst


def block_state(case, seed):
    s = {"in": inputs(case, seed), "w": [], "out": []}
    m = case["m"]
    for layer in range(case["layers"]):
        w = []
        for (op, mats, cols, _, _), raws in zip(steps(case), raw_weights(case, seed, layer)):
            w.append([to_slab(t, r, rows, cols) for (t, rows, _), r in zip(mats * 2, raws)])
        s["w"].append(w)
        s["out"].append({y: torch.empty((m, rows), dtype=torch.float32, device="cuda")
                         for _, mats, _, _, _ in steps(case) for _, rows, y in mats})
    plan, x = steps(case), s["in"]

    def forward():
        for w, out in zip(s["w"], s["out"]):
            for (op, mats, cols, name, norm), ws in zip(plan, w):
                a = out[name] if name == "act" else x[name]
                nw = x[name + ".norm"] if norm else None
                if op == "group":
                    segs = [(hl.DType[t], wi, rows, out[y]) for (t, rows, y), wi in zip(mats, ws)]
                    (hl.gemm_group if m > 8 else hl.gemv_group)(segs, a, cols, m, norm_w=nw, norm_eps=EPS)
                elif op == "gate_up":
                    t, rows, y = mats[0]
                    hl.gate_up_swiglu(hl.DType[t], ws[0], ws[1], a, out[y], rows, cols, m, norm_w=nw, norm_eps=EPS)
                else:
                    t, rows, y = mats[0]
                    hl.gemv(hl.DType[t], ws[0], a, out[y], rows, cols, m, norm_w=nw, norm_eps=EPS)
        return s["out"]

    s["run"] = captured(forward, s) if case["graph"] else forward
    return s


_stream = None


def captured(forward, s):
    """forward as a graph, captured on one side stream for all states (the library keeps a workspace per stream)."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    _stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(_stream):
        forward()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=_stream):
        forward()
    s["graph"] = g

    def replay():
        g.replay()
        return s["out"]

    return replay


def norm64(x, w):
    return x * torch.rsqrt((x * x).mean(1, keepdim=True) + EPS) * w


def times64(x, t, raw, cols):
    """x W^T in 64 bits, over slices of W's rows."""
    return torch.cat([x @ dequant64(t, raw[r:r + 8192], cols).T for r in range(0, raw.shape[0], 8192)], 1)


def block_exact(case, seed):
    x, res = {k: v.double() for k, v in inputs(case, seed).items()}, []
    for layer in range(case["layers"]):
        out = {}
        for (op, mats, cols, name, norm), raws in zip(steps(case), raw_weights(case, seed, layer)):
            a = out[name] if name == "act" else x[name]
            a = norm64(a, x[name + ".norm"]) if norm else a
            if op == "gate_up":
                t, _, y = mats[0]
                g = times64(a, t, raws[0], cols)
                out[y] = g * torch.sigmoid(g) * times64(a, t, raws[1], cols)
            else:
                for (t, _, y), r in zip(mats, raws):
                    out[y] = times64(a, t, r, cols)
        res.append(out)
    return res


# ---- the other pieces ---------------------------------------------------------------------------------------------


def head_inputs(case, seed):
    x, nw = normal(generator(seed, 1), case["m"], case["cols"]), 1 + 0.1 * normal(generator(seed, 2), case["cols"])
    return x, nw, gguf(case["type"], case["rows"], case["cols"], generator(seed, 3))


def embed_inputs(case, seed):
    raw = gguf(case["type"], case["vocab"], case["cols"], generator(seed, 3))
    ids = torch.randint(0, case["vocab"], (case["m"],), generator=generator(seed, 1), device="cuda").int()
    return raw, ids, 1 + 0.1 * normal(generator(seed, 2), case["cols"])


def gguf_inputs(case, seed):
    x = normal(generator(seed, 1), case["m"], case["cols"])
    return x, [gguf(case["type"], case["rows"], case["cols"], generator(seed, 3, i)) for i in range(case["layers"])]


def prepare(case, seed):
    k = case["kind"]
    if k in ("proj", "layer", "ffn", "mixer"):
        return block_state(case, seed)
    t = hl.DType[case["type"]]
    if k == "head":
        rows, cols, m = case["rows"], case["cols"], case["m"]
        x, nw, raw = head_inputs(case, seed)
        w = to_slab(case["type"], raw, rows, cols)
        del raw
        res = torch.empty((m, 3), dtype=torch.int32, device="cuda")
        ids = torch.empty(m, dtype=torch.int32, device="cuda")
        logits = torch.empty((m, rows), dtype=torch.float32, device="cuda")

        def head():
            hl.lm_head(t, w, x, res, rows, cols, m, logits=logits, valid_rows=case["valid"], ids=ids, norm_w=nw, norm_eps=EPS)
            return {"ids": ids, "logits": logits}

        return {"run": head}
    if k == "embed":
        n, cols, m = case["vocab"], case["cols"], case["m"]
        raw, ids, nw = embed_inputs(case, seed)
        layout = hl.Layout.SLAB if case["layout"] == "slab" else hl.Layout.GGUF
        table = to_slab(case["type"], raw, n, cols) if case["layout"] == "slab" else raw
        del raw
        status = torch.zeros(1, dtype=torch.int32, device="cuda")
        rows, normed = (torch.empty((m, cols), dtype=torch.float32, device="cuda") for _ in range(2))

        def embed():
            hl.get_rows(t, layout, table, n, cols, ids, m, rows, status=status, status_keep=True)
            hl.rms_norm(rows, nw, normed, m, cols, eps=EPS)
            return {"rows": rows, "normed": normed}

        return {"run": embed}
    if k == "gguf":
        rows, cols, m = case["rows"], case["cols"], case["m"]
        x, ws = gguf_inputs(case, seed)
        ys = [torch.empty((m, rows), dtype=torch.float32, device="cuda") for _ in ws]

        def rowwise():
            for w, y in zip(ws, ys):
                hl.gemv(t, w, x, y, rows, cols, m, layout=hl.Layout.GGUF)
            return ys

        return {"run": rowwise}
    # load: the weights lie in pageable host memory
    hidden, inner, td = case["hidden"], case["inner"], hl.DType[case["down"]]
    gate, up = (gguf(case["type"], inner, hidden, generator(seed, 3, i)).cpu().numpy() for i in range(2))
    down = gguf(case["down"], hidden, inner, generator(seed, 3, 2)).cpu().numpy()
    fused = torch.empty(hl.slab_bytes(t, 2 * inner, hidden), dtype=torch.uint8, device="cuda")
    dst = torch.empty(hl.slab_bytes(td, hidden, inner), dtype=torch.uint8, device="cuda")

    def load():
        hl.upload_tensors([(t, hidden, [(gate, inner), (up, inner)], fused), (td, inner, [(down, hidden)], dst)])
        return {"gate_up": fused, "down": dst}

    return {"run": load}


def run(state):
    return state["run"]()


def exact(case, seed):
    k = case["kind"]
    if k in ("proj", "layer", "ffn", "mixer"):
        return block_exact(case, seed)
    if k == "head":
        x, nw, raw = head_inputs(case, seed)
        return {"ids": None, "logits": times64(norm64(x.double(), nw.double()), case["type"], raw, case["cols"])}
    if k == "embed":
        raw, ids, nw = embed_inputs(case, seed)
        rows = dequant64(case["type"], raw[ids.long()], case["cols"])
        return {"rows": rows, "normed": norm64(rows, nw.double())}
    if k == "gguf":
        x, ws = gguf_inputs(case, seed)
        return [times64(x.double(), case["type"], w, case["cols"]) for w in ws]
    return None  # load moves bytes


def work(case):
    k = case["kind"]
    if k in ("proj", "layer", "ffn", "mixer"):
        nbytes = flops = 0
        for op, mats, cols, _, _ in steps(case):
            n = 2 if op == "gate_up" else 1
            nbytes += 4 * case["m"] * cols
            for t, rows, _ in mats:
                nbytes += n * rows * row_bytes(t, cols) + 4 * case["m"] * rows
                flops += 2 * n * case["m"] * rows * cols
        return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}
    if k == "embed":
        return {"bytes": case["m"] * (row_bytes(case["type"], case["cols"]) + 8 * case["cols"]), "flops": 4 * case["m"] * case["cols"]}
    if k == "load":
        n = 2 * case["inner"] * row_bytes(case["type"], case["hidden"]) + case["hidden"] * row_bytes(case["down"], case["inner"])
        return {"bytes": 2 * n, "flops": 0}
    layers, m, rows, cols = case.get("layers", 1), case["m"], case["rows"], case["cols"]
    return {"bytes": layers * (rows * row_bytes(case["type"], cols) + 4 * m * (rows + cols)), "flops": layers * 2 * m * rows * cols}


def tolerance(case):
    k = case["kind"]
    # bytes, and results that are defined bit by bit (the CPU's order of additions)
    if k in ("load", "embed", "gguf"):
        return "exact"
    # bf16 operands from 5 rows (gate and up) or 9: two roundings of 2^-9 in each product, again in the product after it
    if k != "head" and case["m"] > (4 if k in ("ffn", "layer") else 8):
        return {"rel": 1e-2, "max": 0.1}
    # sums of 32-bit products in another order
    return {"rel": 3e-6, "max": 3e-5}
