"""The workloads that this library's speed is judged by: quantized matrix products as a
transformer's inference calls them, through the public binding (arcint_amd.qmm).

A case is a dict of an "op" and its sizes:

  mm        one product (MUL_MAT): type, m, k, n columns
  attn      an attention block's four projections in one graph (Q, K and V of one input, then
            the output projection of another): type, hidden, q_rows, kv_rows, o_cols, n
  ffn       a dense FFN block: gate + up + SwiGLU, then down: type, down_type, hidden, ffn, n
  moe       a MoE FFN block from the router's logits on, in one call: type, hidden, ffn, experts,
            top_k, tokens, shared (a gated shared expert)
  moe_ops   the same block (no shared expert) as a program runs it when the experts average many
            tokens: router, gate + up + SwiGLU, down, combine, one call each

Weights are GGUF blocks whose values look like a trained matrix's (centred, about 0.02 rms),
activations are normal with a few large channels, router logits are normal.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from arcint_amd import qmm

TYPES = {"Q4_0": qmm.Q4_0, "Q8_0": qmm.Q8_0, "Q4_K": qmm.Q4_K, "Q5_K": qmm.Q5_K, "Q6_K": qmm.Q6_K,
         "IQ4_NL": qmm.IQ4_NL, "IQ4_XS": qmm.IQ4_XS}
BLOCK = {"Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210),
         "IQ4_NL": (32, 18), "IQ4_XS": (256, 136)}
#: types whose activations are quantized in blocks of 32 (q8_0); the others' in blocks of 256 (q8_K)
BY_32 = ("Q4_0", "Q8_0", "IQ4_NL")
CODEBOOK = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


# ---- the cases ----------------------------------------------------------------------------------

def listed():
    return [
        # Decode, the smallest call: one 4096 x 4096 projection of a 7B-class model for one token.
        # Launch, one memory round trip and the host's call are most of it.
        dict(name="proj_q4_0_n1", op="mm", type="Q4_0", m=4096, k=4096, n=1),
        # Decode: the attention projections of a 27B-class layer (grouped K and V heads: 1024 rows
        # beside 12288) as one graph, so that one activation quantization serves Q, K and V.
        dict(name="attn_q5_k_n1", op="attn", type="Q5_K", hidden=5120, q_rows=12288, kv_rows=1024, o_cols=6144, n=1),
        # Decode: the FFN of that layer, the most common Q4_K_M mix (Q6_K down), weights from HBM.
        dict(name="ffn_q4_k_n1", op="ffn", type="Q4_K", down_type="Q6_K", hidden=5120, ffn=17408, n=1),
        # Decode: the output head over a 152k vocabulary, the largest single stream of a token.
        dict(name="head_q6_k_n1", op="mm", type="Q6_K", m=151936, k=5120, n=1),
        # Decode of eight sequences at once (or a speculative draft's check) on an 8B-class FFN.
        dict(name="ffn_iq4_xs_n8", op="ffn", type="IQ4_XS", down_type="IQ4_XS", hidden=4096, ffn=14336, n=8),
        # A short prompt, an odd number of tokens: between the decode and the prefill kernels.
        dict(name="ffn_q4_k_n77", op="ffn", type="Q4_K", down_type="Q6_K", hidden=5120, ffn=17408, n=77),
        # Ragged in every size: rows not a multiple of the 64-row tile, K not a multiple of 256,
        # an odd number of columns (a small model with a hidden size of 2880).
        dict(name="ragged_q8_0_n203", op="mm", type="Q8_0", m=5761, k=2880, n=203),
        # Prefill: one micro-batch of 512 tokens through the 27B-class FFN.
        dict(name="ffn_q4_k_n512", op="ffn", type="Q4_K", down_type="Q6_K", hidden=5120, ffn=17408, n=512),
        # Prefill, the largest: 2048 tokens through a 7B-class FFN.
        dict(name="ffn_q4_0_n2048", op="ffn", type="Q4_0", down_type="Q4_0", hidden=4096, ffn=11008, n=2048),
        # MoE decode: one token, 10 of 512 experts and the shared expert.
        dict(name="moe_q4_k_t1", op="moe", type="Q4_K", hidden=2048, ffn=512, experts=512, top_k=10, tokens=1,
             shared=True),
        # MoE with 256 tokens in flight: nearly every expert is read, for five tokens each.
        dict(name="moe_q4_k_t256", op="moe", type="Q4_K", hidden=2048, ffn=512, experts=512, top_k=10, tokens=256,
             shared=True),
        # MoE prefill: 1024 tokens over 128 experts, 64 tokens each: grouped products.
        dict(name="moe_q4_k_t1024", op="moe_ops", type="Q4_K", hidden=2048, ffn=512, experts=128, top_k=8,
             tokens=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: every type, 1 to 2048 columns, matrices from 256 x 512 up
    to an output head's half, odd sizes among them."""
    cap = 3 * 2 * 4096 * 11008 * 2048 / 2              # half the largest listed case's operations
    while True:
        t = rng.choice(sorted(TYPES))
        op = rng.choice(("mm", "mm", "mm", "ffn", "ffn", "moe", "moe_ops"))
        if op == "mm":
            k = _log(rng, 512, 17408)
            k -= k % (32 if t in BY_32 else 256)
            c = dict(op=op, type=t, m=_log(rng, 256, 65536), k=k, n=_log(rng, 1, 2048))
            if c["m"] * k > 65536 * 5120:
                continue
        elif op == "ffn":
            c = dict(op=op, type=t, down_type=rng.choice((t, t, "Q6_K")), hidden=256 * _log(rng, 2, 28),
                     ffn=256 * _log(rng, 3, 72), n=_log(rng, 1, 2048))
        else:
            experts = rng.choice((8, 16, 32, 60, 64, 128, 160, 256, 512))
            c = dict(op=op, type=t, hidden=256 * _log(rng, 2, 16), ffn=256 * _log(rng, 2, 8), experts=experts,
                     top_k=rng.randint(2, 10) if experts > 16 else 2, tokens=_log(rng, 1, 1024))
            if c["hidden"] * c["ffn"] * experts > 2048 * 512 * 512:
                continue
            # the one-call block is for experts of few tokens each, the separate ops for many
            if (op == "moe") != (c["tokens"] * c["top_k"] < 32 * experts):
                continue
            if op == "moe":
                c["shared"] = rng.random() < 0.5
        if work(c)["flops"] <= cap:
            return c


# ---- inputs -------------------------------------------------------------------------------------

def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt * 7919 + 12345) % (1 << 62))
    return g


def _f16(v):
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(v.shape[0], 2)


def _weights(t, rows, k, seed, salt):
    """GGUF blocks [blocks, bytes] (uint8, on the GPU) of a [rows, k] matrix, about 0.02 rms."""
    blck, size = BLOCK[t]
    nb = rows * (k // blck)
    g = _gen(seed, salt)
    b = torch.randint(0, 256, (nb, size), dtype=torch.uint8, device="cuda", generator=g)
    u = 0.5 + torch.rand(nb, device="cuda", generator=g)          # how far a block's scale is from the mean
    if t in ("Q4_0", "IQ4_NL"):
        b[:, 0:2] = _f16(u * (0.02 / 4.6 if t == "Q4_0" else 0.02 / 69))
    elif t == "Q8_0":
        b[:, 0:2] = _f16(u * 0.02 / 73)
    elif t in ("Q4_K", "Q5_K"):
        half = 7.5 if t == "Q4_K" else 15.5
        d = u * 0.02 / (43 * (4.6 if t == "Q4_K" else 9.2))
        b[:, 0:2], b[:, 2:4] = _f16(d), _f16(d * half)             # minimum = half the code range: centred
        s = torch.randint(24, 64, (nb, 8), dtype=torch.uint8, device="cuda", generator=g)
        lo, hi = s[:, :4], s[:, 4:]
        b[:, 4:8] = lo | ((hi >> 4) << 6)                          # scales 0-3, the top bits of 4-7
        b[:, 8:12] = lo | ((hi >> 4) << 6)                         # minima 0-3, the top bits of 4-7
        b[:, 12:16] = (hi & 15) | ((hi & 15) << 4)
    elif t == "Q6_K":
        s = torch.randint(48, 128, (nb, 16), dtype=torch.int16, device="cuda", generator=g)
        sign = torch.randint(0, 2, (nb, 16), dtype=torch.int16, device="cuda", generator=g) * 2 - 1
        b[:, 192:208] = (s * sign).to(torch.int8).view(torch.uint8)
        b[:, 208:210] = _f16(u * 0.02 / (90 * 18.5))
    else:
        b[:, 0:2] = _f16(u * 0.02 / (18.5 * 69))
    return b


def _acts(cols, k, seed, salt):
    """float32 [cols, k]: normal, one channel in a hundred five times as large"""
    g = _gen(seed, salt)
    x = torch.randn(cols, k, device="cuda", generator=g)
    return x * (1.0 + 4.0 * (torch.rand(k, device="cuda", generator=g) < 0.01))


_backend = None


def _be():
    """The process's one context, as a program has it."""
    global _backend
    if _backend is None:
        torch.cuda.init()
        _backend = qmm.Backend(torch.cuda.current_device())
    return _backend


class _Held:
    """A tensor of the library and its buffer, freed with the last reference to it; torch reads it
    in place through __cuda_array_interface__."""

    def __init__(self, type_id, ne, data=None):
        be = _be()
        self.t = be.new_tensor(type_id, ne)
        self.__cuda_array_interface__ = {
            "shape": tuple(reversed(ne)), "typestr": "<i4" if type_id == qmm.I32 else "<f4", "strides": None,
            "data": (qmm.load().qmm_buffer_base(ctypes.c_void_p(self.t.buf.ptr)), False), "version": 2}
        if data is not None:
            be.set_tensor(self.t, data)

    def __del__(self):
        if _backend is not None and _backend.h:
            _backend.free_buffer(self.t.buf)

    def view(self):
        return torch.as_tensor(self, device="cuda")


def _weight(t, ne, seed, salt):
    return _Held(TYPES[t], ne, _weights(t, math.prod(ne[1:]), ne[0], seed, salt).cpu().numpy())


def _input(x, ne=None):
    return _Held(qmm.F32, ne or (x.shape[1], x.shape[0]), x.cpu().numpy())


def _out(*ne, type_id=qmm.F32):
    return _Held(type_id, ne, np.zeros(math.prod(ne), np.int32 if type_id == qmm.I32 else np.float32))


def _logits(case, seed):
    return torch.randn(case["tokens"], case["experts"], device="cuda", generator=_gen(seed, 20))


def prepare(case, seed):
    op, s = case["op"], {"op": case["op"]}
    if op == "mm":
        s["w"] = _weight(case["type"], (case["k"], case["m"]), seed, 1)
        s["x"] = _input(_acts(case["n"], case["k"], seed, 10))
        outs = {"y": _out(case["m"], case["n"])}
    elif op == "attn":
        t, n, h = case["type"], case["n"], case["hidden"]
        s["x"], s["a"] = _input(_acts(n, h, seed, 10)), _input(_acts(n, case["o_cols"], seed, 11))
        outs = {}
        for i, (name, k, m) in enumerate(_projections(case)):
            s["w" + name] = _weight(t, (k, m), seed, 1 + i)
            outs[name] = _out(m, n)
        s["nodes"] = [(qmm.OP_MUL_MAT, s["w" + name].t, s["a" if name == "o" else "x"].t, None, outs[name].t)
                      for name in "qkvo"]
    elif op == "ffn":
        t, n, h, f = case["type"], case["n"], case["hidden"], case["ffn"]
        s["gate"], s["up"] = _weight(t, (h, f), seed, 1), _weight(t, (h, f), seed, 2)
        s["down"] = _weight(case["down_type"], (f, h), seed, 3)
        s["x"] = _input(_acts(n, h, seed, 10))
        outs = {"h": _out(f, n), "y": _out(h, n)}
    else:
        t, n, h, f, e, j = (case[v] for v in ("type", "tokens", "hidden", "ffn", "experts", "top_k"))
        s["gate"], s["up"] = _weight(t, (h, f, e), seed, 1), _weight(t, (h, f, e), seed, 2)
        s["down"] = _weight(t, (f, h, e), seed, 3)
        s["logits"] = _input(_logits(case, seed))
        x = _acts(n, h, seed, 10)
        outs = {"ids": _out(j, n, type_id=qmm.I32), "weights": _out(j, n), "y": _out(h, n)}
        if op == "moe":
            s["x"] = _input(x)
            s["shared"] = s["shared_logit"] = None
            if case["shared"]:
                held = [_weight(t, ne, seed, 4 + i) for i, ne in enumerate(((h, f), (h, f), (f, h)))]
                s["held"], s["shared"] = held, tuple(v.t for v in held)
                s["shared_logit"] = _input(_acts(n, 1, seed, 12))
        else:
            s["x"] = _input(x, (h, 1, n))
            outs["h"] = _out(f, j, n)
            s["expert_out"] = _out(h, j, n)
    s.update(("out_" + name, v) for name, v in outs.items())
    s["outputs"] = {name: v.view() for name, v in outs.items()}
    return s


def _projections(case):
    h = case["hidden"]
    return (("q", h, case["q_rows"]), ("k", h, case["kv_rows"]), ("v", h, case["kv_rows"]), ("o", case["o_cols"], h))


def run(s):
    be, op = _be(), s["op"]
    if op == "mm":
        be.mul_mat(s["w"].t, s["x"].t, s["out_y"].t)
    elif op == "attn":
        be.graph_compute(s["nodes"])
    elif op == "ffn":
        be.mul_mat_glu(s["gate"].t, s["up"].t, s["x"].t, s["out_h"].t)
        be.mul_mat(s["down"].t, s["out_h"].t, s["out_y"].t)
    elif op == "moe":
        be.moe_ffn(s["gate"].t, s["up"].t, s["down"].t, s["x"].t, s["out_ids"].t, s["out_weights"].t, s["out_y"].t,
                   s["shared"], s["shared_logit"].t if s["shared_logit"] else None, logits=s["logits"].t)
    else:
        be.moe_topk(s["logits"].t, s["out_ids"].t, s["out_weights"].t)
        be.mul_mat_id_glu(s["gate"].t, s["up"].t, s["x"].t, s["out_ids"].t, s["out_h"].t)
        be.mul_mat_id(s["down"].t, s["out_h"].t, s["out_ids"].t, s["expert_out"].t)
        be.moe_combine(s["expert_out"].t, s["out_weights"].t, s["out_y"].t)
    return s["outputs"]


# ---- what a pass cannot do without ---------------------------------------------------------------

def _bytes(t, k, m):
    return k // BLOCK[t][0] * BLOCK[t][1] * m


def work(case):
    op = case["op"]
    if op in ("mm", "attn"):
        n = case["n"]
        mats = (("y", case["k"], case["m"]),) if op == "mm" else _projections(case)
        ins = case["k"] if op == "mm" else case["hidden"] + case["o_cols"]
        return {"bytes": sum(_bytes(case["type"], k, m) + 4 * m * n for _, k, m in mats) + 4 * ins * n,
                "flops": sum(2 * k * m * n for _, k, m in mats)}
    h, f = case["hidden"], case["ffn"]
    if op == "ffn":
        n = case["n"]
        return {"bytes": 2 * _bytes(case["type"], h, f) + _bytes(case["down_type"], f, h) + 4 * n * (2 * h + f),
                "flops": 6 * h * f * n}
    n, e, j = case["tokens"], case["experts"], case["top_k"]
    one = 2 * _bytes(case["type"], h, f) + _bytes(case["type"], f, h)
    read = e * (1 - (1 - j / e) ** n)                  # experts that some token chose, on average
    s = 1 if case.get("shared") else 0
    return {"bytes": int((read + s) * one) + 4 * n * (2 * h + e + 2 * j), "flops": 6 * h * f * n * (j + s)}


def tolerance(case):
    """A product of given activations differs by the order of its float32 sums. In a chain, that last
    bit moves an intermediate value across a rounding boundary of the next product's 8-bit
    activations now and then, a whole step of 1/127 of its block's largest value."""
    if case["op"] in ("mm", "attn"):
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 1e-3, "max": 2e-2}


# ---- the same in 64 bits -------------------------------------------------------------------------

def _scale_min(s):
    """the eight 6-bit scales and minima of Q4_K / Q5_K's 12 bytes: two [blocks, 8]"""
    sc = torch.cat((s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)), 1)
    mn = torch.cat((s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)), 1)
    return sc.double(), mn.double()


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _decode(t, b, k):
    """float64 [rows, k] of GGUF blocks [blocks, bytes]"""
    nb = b.shape[0]
    if t in ("Q4_0", "IQ4_NL"):
        q = torch.cat((b[:, 2:] & 15, b[:, 2:] >> 4), 1)
        v = q.double() - 8 if t == "Q4_0" else torch.tensor(CODEBOOK, device=b.device, dtype=torch.float64)[q.long()]
        w = v * _half(b[:, 0:2])
    elif t == "Q8_0":
        w = b[:, 2:].contiguous().view(torch.int8).double() * _half(b[:, 0:2])
    elif t in ("Q4_K", "Q5_K"):
        sc, mn = _scale_min(b[:, 4:16])
        qs = b[:, -128:].reshape(nb, 4, 32)
        q = torch.stack((qs & 15, qs >> 4), 2).reshape(nb, 8, 32).double()
        if t == "Q5_K":
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
            q = q + 16 * ((b[:, 16:48].reshape(nb, 1, 32) >> bit) & 1).double()
        w = (_half(b[:, 0:2]) * sc).unsqueeze(2) * q - (_half(b[:, 2:4]) * mn).unsqueeze(2)
    elif t == "Q6_K":
        ql, qh = b[:, 0:128].reshape(nb, 2, 64), b[:, 128:192].reshape(nb, 2, 32)
        q = torch.stack([((ql[:, :, 32 * (g & 1):32 * (g & 1) + 32] >> (4 * (g >> 1))) & 15)
                         | (((qh >> (2 * g)) & 3) << 4) for g in range(4)], 2).reshape(nb, 16, 16)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (_half(b[:, 208:210]) * sc).unsqueeze(2) * (q.double() - 32)
    else:
        high = b[:, 2].long() | (b[:, 3].long() << 8)
        low = torch.stack((b[:, 4:8] & 15, b[:, 4:8] >> 4), 2).reshape(nb, 8).long()
        at = 2 * torch.arange(8, device=b.device)
        sc = (low | (((high.unsqueeze(1) >> at) & 3) << 4)).double() - 32
        qs = b[:, 8:].reshape(nb, 8, 16)
        q = torch.cat((qs & 15, qs >> 4), 2).long()
        w = (_half(b[:, 0:2]) * sc).unsqueeze(2) * torch.tensor(CODEBOOK, device=b.device, dtype=torch.float64)[q]
    return w.reshape(-1, k)


def _q8(t, x):
    """The 8-bit activations that the products are defined on, as their values in float64: q8_0 (a
    float16 scale for 32) or q8_K (a float32 scale for 256, from the first largest value)."""
    x = x.cpu().float()
    full = torch.tensor(127.0)                         # a tensor: `number / tensor` multiplies by a rounded reciprocal
    if t in BY_32:
        v = x.reshape(-1, 32)
        big = v.abs().amax(1, keepdim=True)
        q = torch.where(big > 0, torch.round(v * (full / big)), torch.zeros_like(v))
        d = (big / 127.0).half().double()
    else:
        v = x.reshape(-1, 256)
        first = v.gather(1, v.abs().argmax(1, keepdim=True))
        inv = -full / first
        q = torch.where(first != 0, torch.round(v * inv).clamp(max=127), torch.zeros_like(v))
        d = torch.where(first != 0, torch.ones_like(inv) / inv, torch.zeros_like(inv)).double()
    return (q.double() * d).reshape(x.shape).cuda()


def _product(t, ne, x, seed, salt):
    """float64 [columns, rows] of the matrix that prepare() gives the same seed and salt"""
    k, m = ne
    b, nb = _weights(t, m, k, seed, salt), k // BLOCK[t][0]
    y = torch.empty(x.shape[0], m, dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // k)                      # half a gigabyte of float64 weights at a time
    for r in range(0, m, step):
        e = min(m, r + step)
        y[:, r:e] = x @ _decode(t, b[r * nb:e * nb], k).t()
    return y


def _silu_mul(g, u):
    return g / (1 + torch.exp(-g)) * u


def exact(case, seed):
    """In 64 bits, a product of given activations with their 8-bit values (that rounding is part of
    what it is), the later products of a chain with unrounded ones (there a last bit decides which
    way a value is rounded, so no rounding of it is the exact one)."""
    op = case["op"]
    if op == "mm":
        x = _q8(case["type"], _acts(case["n"], case["k"], seed, 10))
        return {"y": _product(case["type"], (case["k"], case["m"]), x, seed, 1)}
    if op == "attn":
        t, n = case["type"], case["n"]
        x, a = _q8(t, _acts(n, case["hidden"], seed, 10)), _q8(t, _acts(n, case["o_cols"], seed, 11))
        return {name: _product(t, (k, m), a if name == "o" else x, seed, 1 + i)
                for i, (name, k, m) in enumerate(_projections(case))}
    h, f, t = case["hidden"], case["ffn"], case["type"]
    if op == "ffn":
        x = _q8(t, _acts(case["n"], h, seed, 10))
        mid = _silu_mul(_product(t, (h, f), x, seed, 1), _product(t, (h, f), x, seed, 2))
        return {"h": mid, "y": _product(case["down_type"], (f, h), mid, seed, 3)}
    n, e, j = case["tokens"], case["experts"], case["top_k"]
    p = torch.softmax(_logits(case, seed).double(), 1)
    top, ids = torch.topk(p, j, dim=1)
    wts = top / top.sum(1, keepdim=True).clamp(min=6.103515625e-5)
    x = _q8(t, _acts(n, h, seed, 10))
    gate, up, down = (_weights(t, e * m, k, seed, 1 + i) for i, (k, m) in enumerate(((h, f), (h, f), (f, h))))
    mid = torch.zeros(n, j, f, dtype=torch.float64, device="cuda")
    y = torch.zeros(n, h, dtype=torch.float64, device="cuda")
    for i in range(e):
        tok, slot = (ids == i).nonzero(as_tuple=True)
        if not len(tok):
            continue
        g, u, d = (_decode(t, b.reshape(e, -1, b.shape[1])[i], k) for b, k in ((gate, h), (up, h), (down, f)))
        m = _silu_mul(x[tok] @ g.t(), x[tok] @ u.t())
        mid[tok, slot] = m
        y.index_add_(0, tok, (m @ d.t()) * wts[tok, slot].unsqueeze(1))
    out = {"ids": ids.to(torch.int32), "weights": wts, "y": y}
    if op == "moe_ops":
        out["h"] = mid
    elif case["shared"]:
        m = _silu_mul(_product(t, (h, f), x, seed, 4), _product(t, (h, f), x, seed, 5))
        y += _product(t, (f, h), m, seed, 6) * torch.sigmoid(_acts(n, 1, seed, 12).double())
    return out
