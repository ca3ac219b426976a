"""The work that a GGUF inference engine has this framework do, as measurable cases.

Families (the `family` of a case):
  matvec     one projection of one token, `Backend.matvec` (host arrays, as fastgguf.c's own call
             sites hand them over) or `matvec_dev` (activations resident in device memory)
  layers     a token's dense layers, recorded once as a HIP graph and replayed per token: fused QKV,
             O, and the SiLU FFN of each layer
  matmul     one projection of a batch of 2..64 tokens: prompt reading, and the small batches of a
             prompt's tail or of several sequences
  moe        the mixture-of-experts FFN of 1..64 tokens, the routing included
  attention  one layer's attention over the fp32 KV ring cache, decode and prompt batches
  turbo      the same over the TurboQuant KV cache: the new rows stored, then the attention

Weights are random GGUF blocks with the value distributions of the benchmark, activations N(0, 1).
`exact` decodes the blocks and evaluates every case in float64 with plain torch; where the path
quantizes activations (Q8 / Q8_K blocks: part of what it computes) it quantizes them too.
"""
from __future__ import annotations

import math

import torch

from fastgguf_amd.backend import Backend

# GGUF type: (GGML code, values per block, bytes per block, {byte offset: fp16 scale magnitude})
TYPES = {
    "f32": (0, 1, 4, {}), "f16": (1, 1, 2, {}), "bf16": (30, 1, 2, {}),
    "q4_0": (2, 32, 18, {0: 0.01}), "q4_1": (3, 32, 20, {0: 0.01, 2: 0.05}),
    "q5_0": (6, 32, 22, {0: 0.01}), "q5_1": (7, 32, 24, {0: 0.01, 2: 0.05}), "q8_0": (8, 32, 34, {0: 0.01}),
    "q2_k": (10, 256, 84, {80: 0.004, 82: 0.002}), "q3_k": (11, 256, 110, {108: 0.004}),
    "q4_k": (12, 256, 144, {0: 0.005, 2: 0.005}), "q5_k": (13, 256, 176, {0: 0.005, 2: 0.005}),
    "q6_k": (14, 256, 210, {208: 0.002}), "iq4_nl": (20, 32, 18, {0: 0.01}), "iq4_xs": (23, 256, 136, {0: 0.004}),
}
FLOATS = ("f32", "f16", "bf16")
Q8K = ("q4_k", "q5_k", "q6_k")  # activations in Q8_K blocks of 256; the other block types in Q8 blocks of 32
IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]
KVQ4 = [-2.7326, -2.0690, -1.6181, -1.2562, -0.9424, -0.6568, -0.3881, -0.1284]
KVQ4 = KVQ4 + [-v for v in reversed(KVQ4)]
KVQ2 = [-1.5104, -0.4528, 0.4528, 1.5104]

_backend = None


def backend() -> Backend:
    """The process's device context: a program opens one and keeps it."""
    global _backend
    if _backend is None:
        _backend = Backend(0)
    return _backend


# ---- the cases ----

def listed():
    return [
        # one host-array projection as the drop-in patch calls it: a square Q8_0 matrix, batch 1
        dict(name="matvec_host_q8_0", family="matvec", type="q8_0", rows=4096, cols=4096, host=True),
        # generation: four Llama-3-8B-shaped Q4_K layers of one token, a quarter GB of weights and more
        dict(name="decode_layers_q4_k", family="layers", type="q4_k", hidden=4096, qkv=6144, ff=14336, layers=4),
        # generation: the logits of one token, a Q6_K output matrix over a 128256-entry vocabulary
        dict(name="lm_head_q6_k", family="matvec", type="q6_k", rows=128256, cols=4096, host=False),
        # prompt reading of a Q4_K_M file: a full batch through the FFN's gate
        dict(name="prompt_q4_k", family="matmul", type="q4_k", rows=14336, cols=4096, tokens=64),
        # the same file's Q6_K down projection, long rows, a prompt's ragged last batch
        dict(name="prompt_q6_k_down", family="matmul", type="q6_k", rows=4096, cols=14336, tokens=45),
        # prompt reading of a Q5_K_M file
        dict(name="prompt_q5_k", family="matmul", type="q5_k", rows=14336, cols=4096, tokens=64),
        # five tokens: a prompt's short tail, or a few drafted tokens checked at once
        dict(name="few_tokens_q4_k", family="matmul", type="q4_k", rows=14336, cols=4096, tokens=5),
        # generation with a 128-expert model, 8 experts a token
        dict(name="moe_decode", family="moe", type="q4_k", experts=128, hidden=2048, ff=768, k=8, tokens=1),
        # its prompt reading
        dict(name="moe_prompt", family="moe", type="q4_k", experts=128, hidden=2048, ff=768, k=8, tokens=64),
        # one token's attention over a 4096-position cache, 32 heads over 8 K / V heads
        dict(name="attention_decode", family="attention", heads=32, kv_heads=8, hd=128, past=4095, tokens=1),
        # a prompt batch's attention late in a long prompt
        dict(name="attention_prompt", family="attention", heads=32, kv_heads=8, hd=128, past=4032, tokens=64),
        # one token's cache write and attention over the 4-bit K / 4-bit V cache
        dict(name="turbo_decode", family="turbo", heads=32, kv_heads=8, hd=128, past=4095, tokens=1, kbits=4, vbits=4),
    ]


def _log(rng, lo, hi):
    """An integer of lo..hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _tokens(rng):
    """A batch of 2..64 tokens: small ones, whole prompt batches, and everything between."""
    return rng.choice([_log(rng, 2, 7), rng.randint(8, 64), rng.randint(8, 64), 64])


def draw(rng):
    family = rng.choice(["matvec", "matvec", "layers", "matmul", "matmul", "matmul", "moe", "attention", "attention", "turbo"])
    if family in ("matvec", "matmul"):
        t = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "q5_k"] + list(TYPES))
        unit = TYPES[t][1] if t not in FLOATS else 8
        cols = max(unit, _log(rng, 1024, 16384) // unit * unit)
        # at most 24 M weights: every drawn projection stays below the listed largest ones
        rows = _log(rng, 256, min(32768, 24_000_000 // cols))
        rows = rows if rng.random() < 0.3 else max(8, rows // 8 * 8)
        case = dict(family=family, type=t, rows=rows, cols=cols)
        if family == "matvec":
            case["host"] = rng.random() < 0.4
        else:
            case["tokens"] = _tokens(rng)
        return case
    if family == "layers":
        hidden = rng.randint(4, 18) * 256
        ff = max(256, int(hidden * rng.uniform(2.5, 3.5)) // 256 * 256)
        kv = hidden // rng.choice([1, 4, 8]) // 64 * 64
        return dict(family="layers", type=rng.choice(["q4_k", "q4_k", "q5_k", "q6_k", "q8_0", "q4_0", "iq4_xs"]), hidden=hidden,
                    qkv=hidden + 2 * kv, ff=ff, layers=rng.randint(1, 3))
    if family == "moe":
        experts = rng.choice([8, 16, 32, 60, 64, 128])
        return dict(family="moe", type=rng.choice(["q4_k", "q4_k", "q4_k", "q5_k", "q8_0"]), experts=experts, hidden=rng.randint(4, 8) * 256,
                    ff=rng.randint(1, 3) * 256, k=rng.choice([2, 4, 6, 8]), tokens=rng.choice([1, 1, 64, rng.randint(2, 64)]))
    kv_heads = rng.choice([1, 2, 4, 8])
    heads = kv_heads * rng.choice([1, 2, 4, 8]) if kv_heads < 8 else kv_heads * rng.choice([1, 2, 4])
    tokens = rng.choice([1, 1, 64, rng.randint(2, 64)])
    past = _log(rng, 16, 4096 if tokens > 1 else 8192)
    case = dict(family=family, heads=heads, kv_heads=kv_heads, past=past, tokens=tokens)
    if family == "attention":
        return dict(case, hd=rng.choice([64, 80, 96, 128, 128, 256 if tokens < 16 else 128]))
    return dict(case, hd=rng.choice([64, 128, 128]), kbits=rng.choice([4, 8]), vbits=rng.choice([2, 4, 4, 8]))


# ---- inputs: made on the GPU from the seed, the same for prepare() and exact() ----

def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000 + what)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _weights(t, rows, cols, g):
    """A random matrix in GGUF blocks: uint8 [rows, row bytes] on the GPU."""
    if t in FLOATS:
        w = _normal(g, rows, cols) * 0.02
        return w.to({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[t]).view(torch.uint8).reshape(rows, -1)
    _, per, size, scales = TYPES[t]
    n = rows * (cols // per)
    blk = torch.randint(0, 256, (n, size), generator=g, device="cuda", dtype=torch.uint8)
    for at, mag in scales.items():
        d = _normal(g, n, 1) * mag
        if not (at == 2 and t in ("q4_1", "q5_1")):  # their minimum takes either sign
            d = d.abs()
        blk[:, at:at + 2] = d.half().view(torch.uint8)
    if t == "q6_k":  # int8 sub-block scales in [-64, 63]
        blk[:, 192:208] = torch.randint(-64, 64, (n, 16), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
    if t == "q8_0":  # quants in [-127, 127]
        blk[:, 2:34] = torch.randint(-127, 128, (n, 32), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
    return blk.reshape(rows, -1)


def _layer_shapes(c):
    return [("qkv", c["qkv"], c["hidden"]), ("o", c["hidden"], c["hidden"]), ("gate", c["ff"], c["hidden"]),
            ("up", c["ff"], c["hidden"]), ("down", c["hidden"], c["ff"])]


def _inputs(case, seed):
    """Every input of a case, by name: weights (block bytes) and fp32 / int tensors on the GPU."""
    f = case["family"]
    if f in ("matvec", "matmul"):
        return {"w": _weights(case["type"], case["rows"], case["cols"], _gen(seed, 1)),
                "x": _normal(_gen(seed, 2), case.get("tokens", 1), case["cols"])}
    if f == "layers":
        got = {}
        for n in range(case["layers"]):
            for k, (name, rows, cols) in enumerate(_layer_shapes(case)):
                got[f"{name}{n}"] = _weights(case["type"], rows, cols, _gen(seed, 10 + 10 * n + k))
            got[f"x{n}"] = _normal(_gen(seed, 18 + 10 * n), 3, case["hidden"])  # the inputs of QKV, O and the FFN
        return got
    if f == "moe":
        e, h, ff, n = case["experts"], case["hidden"], case["ff"], case["tokens"]
        return {"gate": _weights(case["type"], e * ff, h, _gen(seed, 1)), "up": _weights(case["type"], e * ff, h, _gen(seed, 2)),
                "down": _weights(case["type"], e * h, ff, _gen(seed, 3)), "x": _normal(_gen(seed, 4), n, h),
                "logits": _normal(_gen(seed, 5), n, e)}
    n, hd, kv = case["tokens"], case["hd"], case["kv_heads"]
    cap = case["past"] + n
    en = torch.arange(case["past"], cap, device="cuda", dtype=torch.int32)  # token t sees positions 0..past + t
    got = {"q": _normal(_gen(seed, 1), n, case["heads"], hd), "st": torch.zeros_like(en), "en": en}
    if f == "attention":
        return dict(got, k=_normal(_gen(seed, 2), cap, kv, hd), v=_normal(_gen(seed, 3), cap, kv, hd))
    got.update(kn=_normal(_gen(seed, 2), n, kv, hd), vn=_normal(_gen(seed, 3), n, kv, hd))
    for name, bits, what in (("kq", case["kbits"], 4), ("vq", case["vbits"], 5)):  # the records of the past
        got[name] = _kvq_records(_normal(_gen(seed, what), cap, kv, hd), bits)
    return got


# ---- prepare / run ----

class State:
    """What a program keeps: tensors on the device, buffers, a recorded graph. Freed with the object."""

    def __init__(self, case, call, outputs, tensors=(), graph=None, keep=None):
        self.case, self.call, self.outputs = case, call, outputs
        self.tensors, self.graph, self.keep = list(tensors), graph, keep

    def __del__(self):
        try:
            if self.graph is not None:
                _backend.graph_destroy(self.graph)
            for t in self.tensors:
                t.free()
        except Exception:  # the interpreter is going down
            pass


def _upload(t, w, rows, cols, n_mats=1, order=-1):
    return backend().upload(TYPES[t][0], cols, w.cpu().numpy().reshape(-1), rows=rows, n_mats=n_mats, order=order)


def prepare(case, seed):
    be, f, i = backend(), case["family"], _inputs(case, seed)
    if f in ("matvec", "matmul"):
        rows, n = case["rows"], case.get("tokens", 1)
        w = _upload(case["type"], i["w"], rows, case["cols"])
        if f == "matvec" and case["host"]:
            x = i["x"][0].cpu().numpy()
            return State(case, lambda: be.matvec(w, x), None, [w])
        x, y = i["x"], torch.empty(n, rows, device="cuda")
        torch.cuda.synchronize()
        if f == "matvec":
            return State(case, lambda: be.matvec_dev(w, x.data_ptr(), y.data_ptr()), y[0], [w], keep=x)
        return State(case, lambda: be.matmul_dev(w, x.data_ptr(), y.data_ptr(), n), y, [w], keep=x)
    if f == "layers":
        tensors, out = [], {}
        for n in range(case["layers"]):
            tensors += [_upload(case["type"], i.pop(f"{name}{n}"), rows, cols) for name, rows, cols in _layer_shapes(case)]
            out.update({f"qkv{n}": torch.empty(case["qkv"], device="cuda"), f"o{n}": torch.empty(case["hidden"], device="cuda"),
                        f"h{n}": torch.empty(case["ff"], device="cuda"), f"y{n}": torch.empty(case["hidden"], device="cuda")})
        torch.cuda.synchronize()

        def token():
            for n in range(case["layers"]):
                qkv, o, gate, up, down = tensors[5 * n:5 * n + 5]
                x = i[f"x{n}"]
                be.matvec_dev(qkv, x[0].data_ptr(), out[f"qkv{n}"].data_ptr())
                be.matvec_dev(o, x[1].data_ptr(), out[f"o{n}"].data_ptr())
                be.ffn_dev(gate, up, down, x[2].data_ptr(), out[f"h{n}"].data_ptr(), out[f"y{n}"].data_ptr())

        token()  # sizes the context's scratch, as a program does before it records
        be.sync()
        be.graph_begin()
        token()
        g = be.graph_end()
        return State(case, lambda: be.graph_launch(g), out, tensors, graph=g, keep=i)
    if f == "moe":
        t, e, h, ff = case["type"], case["experts"], case["hidden"], case["ff"]
        gate, up = _upload(t, i.pop("gate"), ff, h, e), _upload(t, i.pop("up"), ff, h, e)
        down = _upload(t, i.pop("down"), h, ff, e)
        y, x, lg = torch.empty(case["tokens"], h, device="cuda"), i["x"], i["logits"]
        torch.cuda.synchronize()
        return State(case, lambda: be.moe_ffn_dev(gate, up, down, case["k"], lg.data_ptr(), x.data_ptr(), y.data_ptr(), case["tokens"]),
                     y, [gate, up, down], keep=i)
    n, hd, nh, kv = case["tokens"], case["hd"], case["heads"], case["kv_heads"]
    cap, scale = case["past"] + n, 1.0 / math.sqrt(hd)
    o = torch.empty(n, nh, hd, device="cuda")
    p = {k: v.data_ptr() for k, v in i.items()}
    torch.cuda.synchronize()
    if f == "attention":
        return State(case, lambda: be.attention_dev(n, nh, kv, hd, p["q"], o.data_ptr(), p["k"], p["v"], kv * hd, cap, p["st"], p["en"],
                                                    cap, scale), o, keep=i)
    kb, vb = case["kbits"], case["vbits"]

    def step():
        be.kvq_store_dev(n, kv, hd, kb, vb, p["kn"], p["vn"], kv * hd, p["kq"], p["vq"], cap, p["en"])
        be.kvq_attention_dev(n, nh, kv, hd, kb, vb, p["q"], o.data_ptr(), p["kq"], p["vq"], cap, p["st"], p["en"], cap, scale)

    return State(case, step, {"o": o, "kq": i["kq"], "vq": i["vq"]}, keep=i)


def run(state):
    r = state.call()
    return r if state.outputs is None else state.outputs


# ---- work and tolerance ----

def _mat_bytes(t, rows, cols):
    return rows * (cols // TYPES[t][1]) * TYPES[t][2]


def work(case):
    f = case["family"]
    if f in ("matvec", "matmul"):
        n, rows, cols = case.get("tokens", 1), case["rows"], case["cols"]
        return {"bytes": _mat_bytes(case["type"], rows, cols) + 4 * n * (rows + cols), "flops": 2 * n * rows * cols}
    if f == "layers":
        s = _layer_shapes(case)
        return {"bytes": case["layers"] * sum(_mat_bytes(case["type"], r, c) + 4 * (r + c) for _, r, c in s),
                "flops": case["layers"] * sum(2 * r * c for _, r, c in s)}
    if f == "moe":
        e, h, ff, k, n = (case[x] for x in ("experts", "hidden", "ff", "k", "tokens"))
        hit = e * (1 - (1 - k / e) ** n)  # experts that some token selects, on average
        per = 2 * _mat_bytes(case["type"], ff, h) + _mat_bytes(case["type"], h, ff)
        return {"bytes": hit * per + 4 * n * (2 * h + e), "flops": 6 * n * k * h * ff}
    n, hd, nh, kv, past = (case[x] for x in ("tokens", "hd", "heads", "kv_heads", "past"))
    keys = past + (n + 1) / 2
    flops = 4 * n * nh * hd * keys
    if f == "attention":
        return {"bytes": 4 * (2 * (past + n) * kv * hd + 2 * n * nh * hd), "flops": flops}
    rec = 8 + hd * (case["kbits"] + case["vbits"]) // 8
    return {"bytes": (past + n) * kv * rec + 4 * (2 * n * nh * hd + 2 * n * kv * hd) + n * kv * rec, "flops": flops}


def tolerance(case):
    f = case["family"]
    if f in ("matvec", "matmul"):
        # fp32 sums of exact integer products: 8e-8 to 6e-7 from float64 (bf16: one fp32 chain per row)
        return {"rel": 1e-5} if case["type"] == "bf16" else {"rel": 2e-6}
    if f in ("layers", "moe"):
        # h = silu(g) u is quantized to 8 bits again: where a last-bit difference of h moves one quant by
        # one, an output row moves by about 1 / (40 sqrt(ff)) of its size
        return {"rel": 5e-4, "max": 0.02}
    return {"rel": 5e-6}  # 1.2e-6 from float64; the cache records of `turbo` are bytes and stay the same


# ---- float64 ----

def _halves(blk, at):
    return blk[:, at:at + 2].contiguous().view(torch.float16).double()


def _decode(t, w, cols):
    """float64 values [rows, cols] of GGUF blocks."""
    rows = w.shape[0]
    if t in FLOATS:
        return w.contiguous().view({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[t]).double().reshape(rows, cols)
    _, per, size, _ = TYPES[t]
    b = w.reshape(-1, size)
    n = b.shape[0]
    i16 = lambda v: v.to(torch.int16)  # noqa: E731
    if per == 32:
        d = _halves(b, 0)
        if t == "q8_0":
            return (d * b[:, 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
        q = b[:, size - 16:]
        v = i16(torch.cat([q & 15, q >> 4], 1))
        if t in ("q5_0", "q5_1"):
            at = 2 if t == "q5_0" else 4
            bits = (b[:, at:at + 4, None] >> torch.arange(8, device=b.device, dtype=torch.uint8)) & 1
            v = v + 16 * i16(bits.reshape(n, 32))
        if t == "iq4_nl":
            return (d * torch.tensor(IQ4, device=b.device, dtype=torch.float64)[v.long()]).reshape(rows, cols)
        v = v.double()
        if t in ("q4_1", "q5_1"):
            return (d * v + _halves(b, 2)).reshape(rows, cols)
        return (d * (v - (8 if t == "q4_0" else 16))).reshape(rows, cols)
    if t in ("q4_k", "q5_k"):
        s = i16(b[:, 4:16])
        lo, mid, hi = s[:, :4], s[:, 4:8], s[:, 8:]
        sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
        mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
        q = b[:, size - 128:].reshape(n, 4, 1, 32)
        v = i16(torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32))
        if t == "q5_k":
            bits = (b[:, 16:48][:, None, :] >> torch.arange(8, device=b.device, dtype=torch.uint8)[None, :, None]) & 1
            v = v + 16 * i16(bits)
        return ((_halves(b, 0) * sc)[:, :, None] * v - (_halves(b, 2) * mn)[:, :, None]).reshape(rows, cols)
    if t == "q6_k":
        ql, qh = i16(b[:, :128]).reshape(n, 2, 2, 32), i16(b[:, 128:192]).reshape(n, 2, 1, 32)
        nib = torch.cat([ql & 15, ql >> 4], 2)  # [n, 2, 4, 32]
        top = (qh >> torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int16).reshape(1, 1, 4, 1)) & 3
        v = (nib | (top << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return (_halves(b, 208)[:, :, None] * sc[:, :, None] * v.reshape(n, 16, 16)).reshape(rows, cols)
    if t in ("q2_k", "q3_k"):
        q = i16(b[:, 16:80] if t == "q2_k" else b[:, 32:96]).reshape(n, 2, 1, 32)
        v = ((q >> torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int16).reshape(1, 1, 4, 1)) & 3).reshape(n, 16, 16)
        if t == "q2_k":
            s = i16(b[:, :16])
            return ((_halves(b, 80) * (s & 15))[:, :, None] * v - (_halves(b, 82) * (s >> 4))[:, :, None]).reshape(rows, cols)
        bits = (i16(b[:, :32])[:, None, :] >> torch.arange(8, device=b.device, dtype=torch.int16)[None, :, None]) & 1
        v = v - 4 * (1 - bits.reshape(n, 16, 16))
        s = i16(b[:, 96:108])
        low = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
        top = torch.cat([(s[:, 8:] >> (2 * j)) & 3 for j in range(4)], 1)
        return ((_halves(b, 108) * ((low | (top << 4)) - 32))[:, :, None] * v).reshape(rows, cols)
    s = i16(b[:, 4:8])  # iq4_xs
    low = torch.stack([s & 15, s >> 4], 2).reshape(n, 8)
    sh = i16(b[:, 2]).int() | (i16(b[:, 3]).int() << 8)
    top = (sh[:, None] >> (2 * torch.arange(8, device=b.device))) & 3
    q = b[:, 8:].reshape(n, 8, 16)
    v = torch.tensor(IQ4, device=b.device, dtype=torch.float64)[torch.cat([q & 15, q >> 4], 2).long()]
    return ((_halves(b, 0) * ((low | (top << 4)) - 32))[:, :, None] * v).reshape(rows, cols)


def _act(t, x):
    """The activations that a type's products read, in float64: fp32 rows quantized to 8 bits per
    block of 256 or 32 values (scale amax / 127 in fp32, ties to even), or as they are."""
    if t in FLOATS:
        return x.double()
    b = x.float().reshape(-1, 256 if t in Q8K else 32)
    d = b.abs().amax(1, keepdim=True) / 127.0
    inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    return (torch.round(b * inv).double() * d.double()).reshape(x.shape)


def _product(t, w, cols, x):
    """x [n, cols] (already _act) times the matrix, in float64, in pieces that fit."""
    step = max(1, (1 << 27) // cols)
    return torch.cat([x @ _decode(t, w[r:r + step], cols).T.contiguous() for r in range(0, w.shape[0], step)], 1)


def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _kvq_signs(n):
    s, out, mask = 0x243F6A8885A308D3, [], (1 << 64) - 1
    for _ in range(n):
        s ^= s >> 12
        s ^= (s << 25) & mask
        s ^= s >> 27
        out.append(1.0 if ((s * 0x2545F4914F6CDD1D) & mask) >> 63 else -1.0)
    return torch.tensor(out, device="cuda", dtype=torch.float64)


def _hadamard(n):
    h = torch.ones(1, 1, device="cuda", dtype=torch.float64)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(n)


def _kvq_records(x, bits):
    """Cache records [slots, K / V heads, 4 + hd bits / 8] of (rotated) rows: the fp32 scale, then the codes."""
    x = x.double()
    if bits == 8:
        s = x.abs().amax(-1, keepdim=True) / 127.0
        codes = torch.round(x / s).to(torch.int8).view(torch.uint8)
    else:
        c = torch.tensor(KVQ4 if bits == 4 else KVQ2, device=x.device, dtype=torch.float64)
        s = x.square().mean(-1, keepdim=True).sqrt()
        codes = torch.bucketize(x / s, (c[1:] + c[:-1]) / 2).to(torch.uint8)
        per = 8 // bits
        codes = sum(codes[..., j::per] << (bits * j) for j in range(per))
    return torch.cat([s.float().view(torch.uint8), codes.to(torch.uint8)], -1).contiguous()


def _kvq_values(rec, bits, hd):
    s = rec[..., :4].contiguous().view(torch.float32).double()
    q = rec[..., 4:]
    if bits == 8:
        return s * q.contiguous().view(torch.int8).double()
    per = 8 // bits
    codes = torch.stack([(q >> (bits * j)) & ((1 << bits) - 1) for j in range(per)], -1).reshape(*q.shape[:-1], hd)
    return s * torch.tensor(KVQ4 if bits == 4 else KVQ2, device=rec.device, dtype=torch.float64)[codes.long()]


def _attend(q, k, v, past):
    """softmax(q k / sqrt(hd)) v per (token, head): q [n, heads, hd], k / v [positions, K / V heads, hd]."""
    n, heads, hd = q.shape
    group = heads // k.shape[1]
    pos = torch.arange(k.shape[0], device=q.device)
    hide = pos[None, :] > past + torch.arange(n, device=q.device)[:, None]
    out = torch.empty(n, heads, hd, device=q.device, dtype=torch.float64)
    for h in range(heads):
        s = (q[:, h].double() @ k[:, h // group].double().T.contiguous()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(hide, -math.inf), 1) @ v[:, h // group].double()
    return out


def exact(case, seed):
    f, i = case["family"], _inputs(case, seed)
    if f in ("matvec", "matmul"):
        y = _product(case["type"], i["w"], case["cols"], _act(case["type"], i["x"]))
        if f == "matmul":
            return y
        return y[0].cpu().numpy() if case["host"] else y[0]
    if f == "layers":
        t, out = case["type"], {}
        for n in range(case["layers"]):
            x = _act(t, i[f"x{n}"])
            out[f"qkv{n}"] = _product(t, i[f"qkv{n}"], case["hidden"], x[0:1])[0]
            out[f"o{n}"] = _product(t, i[f"o{n}"], case["hidden"], x[1:2])[0]
            h = _silu(_product(t, i[f"gate{n}"], case["hidden"], x[2:3])) * _product(t, i[f"up{n}"], case["hidden"], x[2:3])
            out[f"h{n}"] = h[0]
            out[f"y{n}"] = _product(t, i[f"down{n}"], case["ff"], _act(t, h.float()))[0]
        return out
    if f == "moe":
        t, h, ff, k = case["type"], case["hidden"], case["ff"], case["k"]
        p = torch.softmax(i["logits"].double(), 1)
        w, sel = torch.topk(p, k, 1)
        w = w / w.sum(1, keepdim=True)
        x, y = _act(t, i["x"]), torch.zeros(case["tokens"], h, device="cuda", dtype=torch.float64)
        for e in sel.unique().tolist():
            tok, j = (sel == e).nonzero(as_tuple=True)
            g = _product(t, i["gate"][e * ff:(e + 1) * ff], h, x[tok])
            u = _product(t, i["up"][e * ff:(e + 1) * ff], h, x[tok])
            d = _product(t, i["down"][e * h:(e + 1) * h], ff, _act(t, (_silu(g) * u).float()))
            y.index_add_(0, tok, w[tok, j][:, None] * d)
        return y
    if f == "attention":
        return _attend(i["q"], i["k"], i["v"], case["past"])
    hd, past = case["hd"], case["past"]
    rot = _kvq_signs(hd)[:, None] * _hadamard(hd)  # rows times this = the rotation
    kq, vq = i["kq"], i["vq"]
    kq[past:] = _kvq_records((i["kn"].double() @ rot).float(), case["kbits"])
    vq[past:] = _kvq_records((i["vn"].double() @ rot).float(), case["vbits"])
    o = _attend(i["q"].double() @ rot, _kvq_values(kq, case["kbits"], hd), _kvq_values(vq, case["vbits"], hd), past)
    return {"o": o @ rot.T.contiguous(), "kq": None, "vq": None}
