"""Performance cases: the work an inference engine gives this library.

A dense layer's projections at decode, small-batch and prefill sizes, single
matrices of each weight type (a Q4_K_M file's Q6_K output and down matrices
among them), the routed-expert block of a MoE layer, and the BurnHard MoE
forward. Sizes are those of the repository's benchmark: 8B dense shapes
(4096 -> q/k/v 4096 + 1024 + 1024, 4096 -> 12288 -> 4096, vocabulary 151936),
30B-A3B expert banks (128 experts of 2048 -> 768 -> 2048, top-8) and their
neighbourhood.

Weights are block-quantised here with plain torch from N(0, 0.02) values;
activations are N(0, 1) rows with 1% of their columns eight times as large.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("shannon-prime-burnhard_amd"))
import spq4k  # noqa: E402

Q8_0, Q4_K, Q5_K, Q6_K = spq4k.TYPE_Q8_0, spq4k.TYPE_Q4_K, spq4k.TYPE_Q5_K, spq4k.TYPE_Q6_K
TYPES = {"q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
EPS = 1e-6
_ctx = None


def context():
    global _ctx
    if _ctx is None:
        _ctx = spq4k.Context(0)
    return _ctx


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one projection at decode: the smallest call, latency counts
        {"name": "matvec_q4k", "kind": "matmul", "type": "q4_k", "M": 4096, "K": 4096, "T": 1},
        # the vocabulary projection of a Q4_K_M file at decode
        {"name": "head_q6k", "kind": "matmul", "type": "q6_k", "M": 151936, "K": 4096, "T": 1},
        # a dense layer's projections for one token
        {"name": "layer_t1", "kind": "layer", "embd": 4096, "kv": 1024, "ffn": 12288, "down": "q4_k", "T": 1},
        # a few sequences decoded together, or a speculative draft checked
        {"name": "layer_t5", "kind": "layer", "embd": 4096, "kv": 1024, "ffn": 12288, "down": "q4_k", "T": 5},
        # a short prompt of ragged length, Q6_K down as in half of a Q4_K_M file's layers
        {"name": "layer_t100", "kind": "layer", "embd": 4096, "kv": 1024, "ffn": 12288, "down": "q6_k", "T": 100},
        # a full prompt batch
        {"name": "layer_t512", "kind": "layer", "embd": 4096, "kv": 1024, "ffn": 12288, "down": "q4_k", "T": 512},
        # single matrices of the other types at prompt sizes
        {"name": "down_q6k_t384", "kind": "matmul", "type": "q6_k", "M": 4096, "K": 12288, "T": 384},
        {"name": "up_q5k_t150", "kind": "matmul", "type": "q5_k", "M": 13824, "K": 5120, "T": 150},
        {"name": "proj_q80_t40", "kind": "matmul", "type": "q8_0", "M": 4096, "K": 4096, "T": 40},
        # the routed-expert block: one token, and a prompt batch
        {"name": "moe_t1", "kind": "moe", "E": 128, "used": 8, "embd": 2048, "ffn": 768, "down": "q4_k", "T": 1},
        {"name": "moe_t200", "kind": "moe", "E": 128, "used": 8, "embd": 2048, "ffn": 768, "down": "q6_k", "T": 200},
        # the BurnHard MoE forward (fp32 activations), one token
        {"name": "beast", "kind": "beast", "E": 128, "used": 8, "embd": 2048, "ffn": 768, "type": "q4_k"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["matvec", "matmul", "layer", "moe", "beast"], [2, 4, 4, 2, 1])[0]
    if kind in ("matvec", "matmul"):
        t = rng.choice(sorted(TYPES))
        c = {"kind": "matmul", "type": t}
        # whole blocks a row, any number of rows; now and then a multiple of 16 as models have them
        c["K"] = 32 * _log(rng, 48, 432) if t == "q8_0" else 256 * _log(rng, 4, 54)
        if kind == "matvec":
            c["M"], c["T"] = min(_log(rng, 1000, 152000), 620_000_000 // c["K"]), 1
        else:
            c["M"], c["T"] = min(_log(rng, 1000, 28000), 100_000_000 // c["K"]), _log(rng, 2, 512)
        if rng.random() < 0.6:
            c["M"] = max(16, c["M"] // 16 * 16)
        return c
    if kind == "layer":
        return {"kind": "layer", "embd": 256 * rng.randint(8, 16), "kv": 128 * rng.choice([2, 4, 8]),
                "ffn": 256 * rng.randint(20, 48), "down": rng.choice(["q4_k", "q6_k"]),
                "T": 1 if rng.random() < 0.25 else _log(rng, 2, 512)}
    if kind == "moe":
        return {"kind": "moe", "E": rng.choice([32, 60, 64, 128]), "used": rng.choice([2, 4, 6, 8]),
                "embd": 256 * rng.randint(6, 12), "ffn": 256 * rng.randint(2, 6), "down": rng.choice(["q4_k", "q6_k"]),
                "T": _log(rng, 1, 256)}
    return {"kind": "beast", "E": rng.choice([8, 32, 64, 128]), "used": rng.choice([2, 4, 8]),
            "embd": 256 * rng.randint(6, 16), "ffn": 256 * rng.randint(2, 12), "type": rng.choice(sorted(TYPES))}


# ------------------------------------------- quantised weights in plain torch
def _pack_scales(sc, m):
    """6-bit scales and mins [n, 8] -> the 12 packed bytes of a Q4_K / Q5_K block."""
    a = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    b = m[:, :4] | ((m[:, 4:] >> 4) << 6)
    return torch.cat([a, b, (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)], 1)


def _unpack_scales(s):
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:12] & 15) | ((s[:, :4] >> 6) << 4)], 1)
    m = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    return sc, m


def _f16(x):
    """fp32 [n] -> its fp16 bytes [n, 2]"""
    return x.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _encode(t, w):
    """fp32 rows -> block bytes [n, block bytes] of weight type t (absmax / min-max rounding)."""
    if t == Q8_0:
        w = w.reshape(-1, 32)
        d = (w.abs().amax(1) / 127).to(torch.float16)
        q = torch.round(w / d.float()[:, None]).clamp_(-127, 127).to(torch.int8)
        return torch.cat([d.view(torch.uint8).reshape(-1, 2), q.view(torch.uint8)], 1)
    if t == Q6_K:
        w = w.reshape(-1, 16, 16)
        s = w.abs().amax(2) / 31
        d = (s.amax(1) / 127).to(torch.float16)
        sc = torch.round(s / d.float()[:, None]).clamp_(1, 127)
        q = (torch.round(w / (d.float()[:, None] * sc)[:, :, None]).clamp_(-32, 31) + 32).to(torch.uint8)
        q = q.reshape(-1, 2, 4, 32)          # half, quarter, l
        lo, hi = q & 15, q >> 4
        ql = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], 2)
        qh = hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)
        return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8),
                          d.view(torch.uint8).reshape(-1, 2)], 1)
    top = 15 if t == Q4_K else 31
    w = w.reshape(-1, 8, 32)
    mn = (-w.amin(2)).clamp_(min=0)
    s = (w.amax(2) + mn) / top
    d, dm = (s.amax(1) / 63).to(torch.float16), (mn.amax(1) / 63).to(torch.float16)
    sc = torch.round(s / d.float()[:, None]).clamp_(1, 63)
    m = torch.round(mn / dm.float()[:, None]).clamp_(0, 63)
    q = torch.round((w + (dm.float()[:, None] * m)[:, :, None]) / (d.float()[:, None] * sc)[:, :, None])
    q = q.clamp_(0, top).to(torch.uint8)
    qs = ((q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)).reshape(-1, 128)
    head = [d.view(torch.uint8).reshape(-1, 2), dm.view(torch.uint8).reshape(-1, 2),
            _pack_scales(sc.to(torch.uint8), m.to(torch.uint8))]
    if t == Q5_K:
        bit = (q >> 4).to(torch.int32) << torch.arange(8, device=q.device, dtype=torch.int32)[None, :, None]
        head.append(bit.sum(1).to(torch.uint8))
    return torch.cat(head + [qs], 1)


def _decode(t, b):
    """block bytes -> fp64 values [n, values of a block]"""
    def half(x):
        return x.contiguous().view(torch.float16).double()[:, 0]
    if t == Q8_0:
        return half(b[:, :2])[:, None] * b[:, 2:].contiguous().view(torch.int8).double()
    if t == Q6_K:
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        q = torch.stack([(ql[:, :, h & 1] >> (4 * (h >> 1)) & 15) | ((qh >> (2 * h) & 3) << 4) for h in range(4)], 2)
        q = q.reshape(-1, 16, 16).double() - 32
        return (half(b[:, 208:210])[:, None, None] * sc[:, :, None] * q).reshape(-1, 256)
    sc, m = _unpack_scales(b[:, 4:16])
    qs = (b[:, 16:] if t == Q4_K else b[:, 48:]).reshape(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if t == Q5_K:
        q = q | torch.stack([(b[:, 16:48] >> j & 1) << 4 for j in range(8)], 1)
    d, dm = half(b[:, 0:2])[:, None], half(b[:, 2:4])[:, None]
    return ((d * sc.double())[:, :, None] * q.double() - (dm * m.double())[:, :, None]).reshape(-1, 256)


def _weights(gen, t, rows, K):
    """[rows, bytes of a row] uint8 on the GPU, of N(0, 0.02) values"""
    nb, size = K // spq4k.BLOCK_VALUES[t], spq4k.BLOCK_BYTES[t]
    out = torch.empty(rows, nb * size, dtype=torch.uint8, device="cuda")
    step = max(1, 50_000_000 // K)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        w = torch.randn(n, K, generator=gen, device="cuda") * 0.02
        out[r:r + n] = _encode(t, w).reshape(n, -1)
    return out


def _acts(gen, T, K):
    """[T, K] fp32: N(0, 1), 1% of the columns eight times as large"""
    x = torch.randn(T, K, generator=gen, device="cuda")
    col = torch.rand(K, generator=gen, device="cuda") < 0.01
    return torch.where(col, x * 8, x)


# ----------------------------------------------------------- inputs of a case
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _inputs(case, seed):
    """Everything random of a case, in one order: torch tensors only."""
    g, kind = _gen(seed), case["kind"]
    if kind == "matmul":
        t = TYPES[case["type"]]
        return {"W": _weights(g, t, case["M"], case["K"]), "x": _acts(g, case["T"], case["K"])}
    if kind == "layer":
        n, kv, f, T = case["embd"], case["kv"], case["ffn"], case["T"]
        dt = TYPES[case["down"]]
        return {"q": _weights(g, Q4_K, n, n), "k": _weights(g, Q4_K, kv, n), "v": _weights(g, Q4_K, kv, n),
                "o": _weights(g, Q4_K, n, n), "gate": _weights(g, Q4_K, f, n), "up": _weights(g, Q4_K, f, n),
                "down": _weights(g, dt, n, f), "x": _acts(g, T, n), "att": _acts(g, T, n), "h": _acts(g, T, n),
                "norm1": 1 + 0.1 * torch.randn(n, generator=g, device="cuda"),
                "norm2": 1 + 0.1 * torch.randn(n, generator=g, device="cuda")}
    E, n, f = case["E"], case["embd"], case["ffn"]
    t = Q4_K if kind == "moe" else TYPES[case["type"]]
    dt = TYPES[case["down"]] if kind == "moe" else t
    got = {"gate": _weights(g, t, E * f, n), "up": _weights(g, t, E * f, n), "down": _weights(g, dt, E * n, f)}
    T = case["T"] if kind == "moe" else 1
    logits = torch.randn(T, E, generator=g, device="cuda")
    got["x"] = _acts(g, T, n)
    if kind == "beast":
        got["logits"] = logits[0].contiguous()
        return got
    top = torch.softmax(logits, 1).topk(case["used"], 1)
    got["ids"] = top.indices.to(torch.int32).contiguous()
    got["p"] = (top.values / top.values.sum(1, keepdim=True)).contiguous()
    return got


def prepare(case, seed):
    c, i, kind = context(), _inputs(case, seed), case["kind"]
    s = {"kind": kind, "in": i, "T": case.get("T", 1)}

    def out(*shape):
        return torch.zeros(*shape, device="cuda")

    def wrap(name, M, K, E=1, t=Q4_K):
        s["w_" + name] = c.wrap(i[name].data_ptr(), M, K, E, t)

    T = s["T"]
    if kind == "matmul":
        wrap("W", case["M"], case["K"], 1, TYPES[case["type"]])
        s["y"] = out(T, case["M"])
    elif kind == "layer":
        n, kv, f = case["embd"], case["kv"], case["ffn"]
        for name, M in (("q", n), ("k", kv), ("v", kv), ("o", n), ("gate", f), ("up", f)):
            wrap(name, M, n)
        wrap("down", n, f, 1, TYPES[case["down"]])
        s.update(q=out(T, n), k=out(T, kv), v=out(T, kv), o=out(T, n), hid=out(T, f), y=out(T, n))
    else:
        E, n, f = case["E"], case["embd"], case["ffn"]
        t = Q4_K if kind == "moe" else TYPES[case["type"]]
        wrap("gate", f, n, E, t)
        wrap("up", f, n, E, t)
        wrap("down", n, f, E, TYPES[case["down"]] if kind == "moe" else t)
        s["used"] = case["used"]
        s["y"] = out(T, n)
        if kind == "beast":
            s["ids"] = torch.zeros(case["used"], dtype=torch.int32, device="cuda")
            s["p"] = out(case["used"])
    return s


def run(s):
    c, i, T, kind = context(), s["in"], s["T"], s["kind"]
    if kind == "matmul":
        c.mul_mat_dev(s["w_W"], i["x"].data_ptr(), s["y"].data_ptr(), T)
        return s["y"]
    if kind == "layer":
        c.mul_mat_rms_norm_dev([s["w_q"], s["w_k"], s["w_v"]], i["x"].data_ptr(), i["norm1"].data_ptr(), EPS,
                               [s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr()], T)
        c.mul_mat_dev(s["w_o"], i["att"].data_ptr(), s["o"].data_ptr(), T)
        c.mul_mat_swiglu_dev(s["w_gate"], s["w_up"], i["h"].data_ptr(), i["norm2"].data_ptr(), EPS,
                             s["hid"].data_ptr(), T)
        c.mul_mat_dev(s["w_down"], s["hid"].data_ptr(), s["y"].data_ptr(), T)
        return {k: s[k] for k in ("q", "k", "v", "o", "hid", "y")}
    if kind == "moe":
        c.moe_ffn_dev(s["w_gate"], s["w_up"], s["w_down"], i["ids"].data_ptr(), i["p"].data_ptr(), s["used"], T,
                      i["x"].data_ptr(), s["y"].data_ptr())
        return s["y"]
    c.beast_moe_forward_dev(s["w_gate"], s["w_up"], s["w_down"], i["logits"].data_ptr(), s["used"],
                            i["x"].data_ptr(), s["y"].data_ptr(), s["ids"].data_ptr(), s["p"].data_ptr())
    return {"y": s["y"], "ids": s["ids"], "scores": s["p"]}


# ------------------------------------------------------- work and correctness
def _row_bytes(t, K):
    return K // spq4k.BLOCK_VALUES[t] * spq4k.BLOCK_BYTES[t]


def work(case):
    kind, T = case["kind"], case.get("T", 1)
    if kind == "matmul":
        M, K = case["M"], case["K"]
        return {"bytes": M * _row_bytes(TYPES[case["type"]], K) + 4 * T * (K + M), "flops": 2 * M * K * T}
    n, f = case["embd"], case["ffn"]
    if kind == "layer":
        kv = case["kv"]
        w = (2 * n + 2 * kv + 2 * f) * _row_bytes(Q4_K, n) + n * _row_bytes(TYPES[case["down"]], f)
        acts = 3 * n + (n + 2 * kv) + n + 2 * f + n   # inputs, q/k/v, o, hidden out and in, y
        return {"bytes": w + 4 * T * acts + 8 * n, "flops": 2 * T * (2 * n * n + 2 * kv * n + 3 * f * n)}
    t = Q4_K if kind == "moe" else TYPES[case["type"]]
    dt = TYPES[case["down"]] if kind == "moe" else t
    experts = min(case["E"], case["used"]) if T == 1 else case["E"] * (1 - (1 - case["used"] / case["E"]) ** T)
    w = experts * (2 * f * _row_bytes(t, n) + n * _row_bytes(dt, f))
    return {"bytes": w + 8 * T * n + 8 * T * case["used"], "flops": 6 * T * case["used"] * n * f}


def tolerance(case):
    # fp32 sums of exact integer block products: 1e-7 to 2e-7 against 64 bits
    if case["kind"] == "matmul":
        return {"rel": 1e-6}
    # fp32 activations, products and sums: 3e-7
    if case["kind"] == "beast":
        return {"rel": 2e-6}
    # the hidden rows are quantised to 8 bits again: a last-bit difference of a
    # hidden value now and then moves it to the neighbouring step, and one step
    # of one value of one row is about 4e-4 of that row's result
    return {"rel": 2e-3}


def _quantise(t, x):
    """fp32 rows -> what the format's activation quantiser keeps of them, in 64 bits. The rounding is part
    of the operation (the integer product is of these values), so it is done in fp32 as stated:
    256-value blocks q = round(x * (-127 / max)), d = 1 / (-127 / max), or for Q8_0 weights 32-value blocks
    q = round(x * (127 / |max|)), d = fp16(|max| / 127)."""
    T, K = x.shape
    if t == Q8_0:
        b = x.reshape(-1, 32)
        a = b.abs().amax(1, keepdim=True)
        n = torch.full_like(a, 127)   # tensors on both sides: a division by or of a plain number is not rounded once
        q = torch.round(b * torch.where(a > 0, n / a, torch.zeros_like(a)))
        return (q.double() * (a / n).to(torch.float16).double()).reshape(T, K)
    b = x.reshape(-1, 256)
    m = b.gather(1, b.abs().argmax(1, keepdim=True))
    s = torch.where(m != 0, torch.full_like(m, -127) / m, torch.zeros_like(m))
    q = torch.round(b * s).clamp_(max=127)
    return (q.double() * torch.where(m != 0, torch.ones_like(s) / s, torch.zeros_like(s)).double()).reshape(T, K)


def _product(t, w, K, x):
    """fp64 [T, rows] = x . decoded rows, a slice of rows at a time"""
    rows = w.shape[0]
    y = torch.empty(x.shape[0], rows, dtype=torch.float64, device="cuda")
    step = max(1, 30_000_000 // K)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        blocks = w[r:r + n].reshape(-1, spq4k.BLOCK_BYTES[t])
        y[:, r:r + n] = x @ _decode(t, blocks).reshape(n, K).t().contiguous()
    return y


def _norm(x, w):
    total = (x * x).double().sum(1, keepdim=True)
    mean = (total / torch.full_like(total, x.shape[1])).float()
    return x * (torch.ones_like(mean) / torch.sqrt(mean + EPS)) * w


def _swiglu(g, u):
    return g / (1 + torch.exp(-g)) * u


def exact(case, seed):
    i, kind = _inputs(case, seed), case["kind"]
    if kind == "matmul":
        t = TYPES[case["type"]]
        return _product(t, i["W"], case["K"], _quantise(t, i["x"]))
    n, f = case["embd"], case["ffn"]
    if kind == "layer":
        dt = TYPES[case["down"]]
        x, h, a = (_quantise(Q4_K, v) for v in (_norm(i["x"], i["norm1"]), _norm(i["h"], i["norm2"]), i["att"]))
        got = {k: _product(Q4_K, i[k], n, x) for k in "qkv"}
        got["o"] = _product(Q4_K, i["o"], n, a)
        got["hid"] = _swiglu(_product(Q4_K, i["gate"], n, h), _product(Q4_K, i["up"], n, h))
        got["y"] = _product(dt, i["down"], f, _quantise(dt, got["hid"].float()))
        return got
    E = case["E"]
    if kind == "moe":
        dt = TYPES[case["down"]]
        ids, p, x = i["ids"].long(), i["p"], _quantise(Q4_K, i["x"])
        y = torch.zeros(case["T"], n, dtype=torch.float64, device="cuda")
        for e in range(E):
            tok, slot = (ids == e).nonzero(as_tuple=True)
            if tok.numel() == 0:
                continue
            w = [i[k].reshape(E, -1, i[k].shape[1])[e] for k in ("gate", "up", "down")]
            hid = _swiglu(_product(Q4_K, w[0], n, x[tok]), _product(Q4_K, w[1], n, x[tok]))
            d = _product(dt, w[2], f, _quantise(dt, hid.float()))
            y.index_add_(0, tok, d * p[tok, slot].double()[:, None])
        return y
    t = TYPES[case["type"]]
    score = torch.softmax(i["logits"].double(), 0).topk(min(case["used"], E))
    p = score.values / score.values.sum()
    y = torch.zeros(n, dtype=torch.float64, device="cuda")
    for e, s in zip(score.indices.tolist(), p):
        w = [i[k].reshape(E, -1, i[k].shape[1])[e] for k in ("gate", "up", "down")]
        x = i["x"].double()
        hid = _swiglu(_product(t, w[0], n, x), _product(t, w[1], n, x))
        y += s * _product(t, w[2], f, hid)[0]
    return {"y": y[None], "ids": None, "scores": p}
