"""The work that a user of this library has it do, as measurable cases.

A chat program decodes token by token (GEMVs over the frozen projections and the LM
head), reads prompts of 2 to 256 tokens at a time, and streams routed experts; a
training program multiplies packed batches of up to 4096 tokens forward and backward.
Weights are quantized blocks (the recipe types q4_K / q5_K / q6_K / q8_0, and the types
that imported bases bring) or fp16 / bf16 rows, around N(0, 0.02); activations are fp32
~N(0, 1).  Shapes are those of a 12B-class decoder layer (hidden 5120, 32 query and 8
key/value heads of 128, ffn 14336) and of a 64-expert layer (hidden 2048, expert ffn
1408), and ranges around them.

Blocks are drawn code by code on the GPU, in the formats' own layouts, so that inputs
are quick to make and the 64-bit results need no decoder of the library.
"""
import math

import torch

import tier_amd

DEV = "cuda"
TYPES = {"q4_0": tier_amd.Q4_0, "q5_0": tier_amd.Q5_0, "q8_0": tier_amd.Q8_0, "q2_K": tier_amd.Q2_K,
         "q3_K": tier_amd.Q3_K, "q4_K": tier_amd.Q4_K, "q5_K": tier_amd.Q5_K, "q6_K": tier_amd.Q6_K,
         "iq4_xs": tier_amd.IQ4_XS, "f16": tier_amd.F16, "bf16": tier_amd.BF16}
#: elements and bytes of a block
BLOCK = {"q4_0": (32, 18), "q5_0": (32, 22), "q8_0": (32, 34), "q2_K": (256, 84), "q3_K": (256, 110),
         "q4_K": (256, 144), "q5_K": (256, 176), "q6_K": (256, 210), "iq4_xs": (256, 136), "f16": (1, 2),
         "bf16": (1, 2)}
IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
RECIPE = ("q4_K", "q5_K", "q6_K", "q8_0")
IMPORTED = ("q4_0", "q5_0", "q2_K", "q3_K", "iq4_xs")


def row_bytes(t, K):
    be, bb = BLOCK[t]
    return K // be * bb


# ------------------------------------------------------------------- inputs
def _codes(g, shape, mid, sd, lo, hi):
    """Integer codes lo..hi as a quantizer of a normal row spreads them."""
    return torch.randn(shape, generator=g, device=DEV).mul_(sd).add_(mid).round_().clamp_(lo, hi).to(torch.int16)


def _scale(g, shape, mid):
    """fp16 block scales within a factor of 1.5 of each other."""
    return (torch.rand(shape, generator=g, device=DEV).mul_(0.4).add_(0.8) * mid).half()


def _ints(g, shape, lo, hi):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=torch.int16)


def _u8(v):
    return v.to(torch.uint8)


def _bytes(h):
    """Last axis of fp16 (or int16) as little-endian bytes."""
    return h.contiguous().view(torch.uint8)


def _kq(g, nb, bits):
    """Codes, 6-bit scales and minima and fp16 d, dmin of nb q4_K / q5_K super-blocks."""
    top = (1 << bits) - 1
    q = _codes(g, (nb, 8, 32), top / 2, top / 5.0, 0, top)
    sc = _ints(g, (nb, 8), 30, 64)
    mn = (sc + _ints(g, (nb, 8), -4, 5)).clamp_(0, 63)
    d = _scale(g, (nb, 1), 0.02 / (top / 5.0 * 46))
    return q, sc, mn, d, (d.float() * (top / 2)).half()


def _kq_head(sc, mn, d, dmin):
    a = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    b = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
    c = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    return [_bytes(d), _bytes(dmin), _u8(a), _u8(b), _u8(c)]


def _kq_value(q, sc, mn, d, dmin):
    return (d.float() * sc)[..., None] * q - (dmin.float() * mn)[..., None]


def weight(t, N, K, g, values=False):
    """N rows of K elements of type t: (bytes [N][row_bytes], fp32 values [N][K] or None)."""
    be, bb = BLOCK[t]
    nb = N * K // be
    v = None
    if t in ("f16", "bf16"):
        w = torch.randn((N, K), generator=g, device=DEV).mul_(0.02).to(torch.float16 if t == "f16" else torch.bfloat16)
        return w, (w.float() if values else None)
    if t == "q8_0":
        q, d = _codes(g, (nb, 32), 0, 42, -127, 127), _scale(g, (nb, 1), 0.02 / 42)
        parts = [_bytes(d), _u8(q & 255)]
        v = d.float() * q if values else None
    elif t == "q4_0":
        q, d = _codes(g, (nb, 32), 8, 3, 0, 15), _scale(g, (nb, 1), 0.02 / 3)
        parts = [_bytes(d), _u8(q[:, :16] | (q[:, 16:] << 4))]
        v = d.float() * (q - 8) if values else None
    elif t == "q5_0":
        q, d = _codes(g, (nb, 32), 16, 6, 0, 31), _scale(g, (nb, 1), 0.02 / 6)
        bit = 1 << torch.arange(8, device=DEV, dtype=torch.int16)
        qh = ((q >> 4).view(nb, 4, 8) * bit).sum(-1)
        parts = [_bytes(d), _u8(qh), _u8((q[:, :16] & 15) | ((q[:, 16:] & 15) << 4))]
        v = d.float() * (q - 16) if values else None
    elif t in ("q4_K", "q5_K"):
        q, sc, mn, d, dmin = _kq(g, nb, 4 if t == "q4_K" else 5)
        p = (q & 15).view(nb, 4, 2, 32)
        qs = _u8(p[:, :, 0] | (p[:, :, 1] << 4)).view(nb, 128)
        parts = _kq_head(sc, mn, d, dmin)
        if t == "q5_K":
            bit = 1 << torch.arange(8, device=DEV, dtype=torch.int16)
            parts.append(_u8(((q >> 4) * bit[:, None]).sum(1)))
        parts.append(qs)
        v = _kq_value(q, sc, mn, d, dmin) if values else None
    elif t == "q6_K":
        q = _codes(g, (nb, 2, 4, 32), 32, 10, 0, 63)
        sc = _ints(g, (nb, 16), 60, 128) * (2 * _ints(g, (nb, 16), 0, 2) - 1)
        d = _scale(g, (nb, 1), 0.02 / (10 * 94))
        ql = (q[:, :, :2] & 15) | ((q[:, :, 2:] & 15) << 4)
        h = q >> 4
        qh = h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)
        parts = [_u8(ql).view(nb, 128), _u8(qh).view(nb, 64), _u8(sc & 255), _bytes(d)]
        v = (d.float() * sc)[..., None] * (q.view(nb, 16, 16) - 32) if values else None
    elif t == "q3_K":
        q = _codes(g, (nb, 8, 32), 3.5, 1.6, 0, 7)
        sc = _ints(g, (nb, 16), 12, 32) * (2 * _ints(g, (nb, 16), 0, 2) - 1)
        d = _scale(g, (nb, 1), 0.02 / (1.6 * 22))
        bit = 1 << torch.arange(8, device=DEV, dtype=torch.int16)
        hm = ((q >> 2) * bit[:, None]).sum(1)
        lo = (q & 3).view(nb, 2, 4, 32)
        qs = lo[:, :, 0] | (lo[:, :, 1] << 2) | (lo[:, :, 2] << 4) | (lo[:, :, 3] << 6)
        s6 = sc + 32
        low = (s6[:, :8] & 15) | ((s6[:, 8:] & 15) << 4)
        h = (s6 >> 4).view(nb, 4, 4)
        high = h[:, 0] | (h[:, 1] << 2) | (h[:, 2] << 4) | (h[:, 3] << 6)
        parts = [_u8(hm), _u8(qs).view(nb, 64), _u8(low), _u8(high), _bytes(d)]
        v = (d.float() * sc)[..., None] * (q.view(nb, 16, 16) - 4) if values else None
    elif t == "q2_K":
        q = _codes(g, (nb, 8, 32), 1.5, 0.9, 0, 3)
        sc = _ints(g, (nb, 16), 8, 16)
        mn = (sc + _ints(g, (nb, 16), -1, 2)).clamp_(0, 15)
        d = _scale(g, (nb, 1), 0.02 / (0.9 * 11))
        dmin = (d.float() * 1.5).half()
        lo = q.view(nb, 2, 4, 32)
        qs = lo[:, :, 0] | (lo[:, :, 1] << 2) | (lo[:, :, 2] << 4) | (lo[:, :, 3] << 6)
        parts = [_u8(sc | (mn << 4)), _u8(qs).view(nb, 64), _bytes(d), _bytes(dmin)]
        v = _kq_value(q.view(nb, 16, 16), sc, mn, d, dmin) if values else None
    elif t == "iq4_xs":
        q = _codes(g, (nb, 8, 32), 7.6, 3.2, 0, 15)
        sc = _ints(g, (nb, 8), 12, 32) * (2 * _ints(g, (nb, 8), 0, 2) - 1)
        d = _scale(g, (nb, 1), 0.02 / (50 * 22))
        s6 = sc + 32
        two = 1 << (2 * torch.arange(8, device=DEV, dtype=torch.int32))
        hi = ((s6 >> 4).int() * two).sum(-1, keepdim=True)
        s4 = (s6 & 15).view(nb, 4, 2)
        parts = [_bytes(d), _u8(hi & 255), _u8(hi >> 8), _u8(s4[:, :, 0] | (s4[:, :, 1] << 4)),
                 _u8(q[:, :, :16] | (q[:, :, 16:] << 4)).view(nb, 128)]
        if values:
            level = torch.tensor(IQ4, device=DEV, dtype=torch.float32)[q.long()]
            v = (d.float() * sc)[..., None] * level
    else:
        raise ValueError(t)
    blocks = torch.cat(parts, 1)
    assert blocks.shape == (nb, bb), (t, blocks.shape)
    return blocks.view(N, row_bytes(t, K)), (v.reshape(N, K) if values else None)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _x(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _y(*shape):
    return torch.zeros(shape, device=DEV)


def _ws(nbytes):
    return torch.empty(max(int(nbytes), 16), dtype=torch.uint8, device=DEV)


def _mul64(x, w):
    """x @ w^T in 64 bits."""
    return x.double() @ w.double().t().contiguous()


def _layer(c):
    """The seven projections of a decoder layer: (type, rows, columns)."""
    H, Q, KV, F = c["hidden"], c["q"], c["kv"], c["ffn"]
    t, v, down = c["type"], c["v"], c["down"]
    return [(t, Q, H), (t, KV, H), (v, KV, H), (t, H, Q), (t, F, H), (t, F, H), (down, H, F)]


# -------------------------------------------------------------------- cases
def listed():
    L12 = {"hidden": 5120, "q": 4096, "kv": 1024, "ffn": 14336}
    return [
        # the smallest call of a decode step: the k projection of one token
        {"name": "gemv_k_proj", "kind": "gemv", "type": "q4_K", "N": 1024, "K": 5120},
        # a projection of an imported base, whose type no recipe of this library makes
        {"name": "gemv_imported", "kind": "gemv", "type": "iq4_xs", "N": 14336, "K": 5120},
        # the LM head of a decode step: dense rows of a vocabulary
        {"name": "lm_head", "kind": "dense", "type": "f16", "N": 32000, "K": 5120},
        # one decoder layer of a decode step, q4_K_M (v and down in q6_K), as a chat program calls it
        {"name": "decode_layer", "kind": "layer", "M": 1, "type": "q4_K", "v": "q6_K", "down": "q6_K", **L12},
        # a short question of a running chat: few tokens against one large projection
        {"name": "prompt_short", "kind": "prompt", "type": "q4_K", "M": 37, "N": 14336, "K": 5120},
        # a full prompt chunk through one decoder layer, q4_K_S (v and down in q5_K)
        {"name": "prompt_chunk", "kind": "layer", "M": 256, "type": "q4_K", "v": "q5_K", "down": "q5_K", **L12},
        # a prompt on an fp16 base: rows kept dense, x split in three parts
        {"name": "prompt_f16", "kind": "rows", "type": "f16", "M": 203, "N": 5120, "K": 4096},
        # a training forward product of a small packed batch on a quantized base
        {"name": "train_fwd", "kind": "train_fwd", "type": "q4_K", "M": 512, "N": 5120, "K": 5120},
        # the backward product of gate and up on a full batch: both weights expanded to
        # fp16, dX = dG Wg, dX += dU Wu (the largest call)
        {"name": "train_dx", "kind": "train_dx", "type": "q4_K", "M": 4096, "N": 14336, "K": 5120},
        # a routed layer over a full batch, and over the eight tokens of a batched decode step
        {"name": "moe_batch", "kind": "moe", "T": 4096, "E": 64, "topk": 8, "hidden": 2048, "ffn": 1408},
        {"name": "moe_decode", "kind": "moe", "T": 8, "E": 64, "topk": 8, "hidden": 2048, "ffn": 1408},
        # the fp32-accurate product of a weight split beforehand, x split on each call
        {"name": "x3s_linear", "kind": "x3s", "M": 4096, "N": 5120, "K": 5120},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, m):
    return max(m, _log(rng, lo, hi) // m * m)


def draw(rng):
    kind = rng.choice(("gemv", "gemv", "dense", "layer", "prompt", "prompt", "rows", "train_fwd", "train_dx", "moe",
                       "moe", "x3s"))
    c = {"kind": kind}
    if kind == "gemv":
        c["type"] = rng.choice(RECIPE if rng.random() < 0.5 else IMPORTED)
        c["N"] = _log(rng, 256, 28672)
        c["K"] = _mult(rng, 1024, 14336, 256)
    elif kind == "dense":
        c["type"] = rng.choice(("f16", "bf16"))
        c["N"] = _log(rng, 4096, 131072)
        c["K"] = _mult(rng, 1024, 8192, 64)
    elif kind == "layer":
        c["M"] = 1 if rng.random() < 0.5 else _log(rng, 2, 256)
        c["type"], c["v"], c["down"] = rng.choice((("q4_K", "q6_K", "q6_K"), ("q4_K", "q4_K", "q4_K"),
                                                   ("q4_K", "q5_K", "q5_K"), ("q5_K", "q6_K", "q6_K"),
                                                   ("q6_K", "q6_K", "q6_K"), ("q8_0", "q8_0", "q8_0")))
        c["hidden"] = _mult(rng, 2048, 6144, 256)
        c["q"] = _mult(rng, 2048, 6144, 256)
        c["kv"] = rng.choice((512, 1024, c["q"]))
        c["ffn"] = _mult(rng, 5632, 16384, 256)
    elif kind == "prompt":
        c["type"] = rng.choice(RECIPE)
        c["M"] = _log(rng, 2, 256)
        c["N"] = _log(rng, 512, 14336)
        c["K"] = _mult(rng, 1024, 14336, 256)
    elif kind == "rows":
        c["type"] = rng.choice(("f16", "bf16"))
        c["M"] = _log(rng, 2, 512)
        c["N"] = _log(rng, 512, 14336)
        c["K"] = _mult(rng, 1024, 14336, 32)
    elif kind == "train_fwd":
        c["type"] = rng.choice(RECIPE)
        c["M"] = _log(rng, 128, 4096)
        c["N"] = _log(rng, 1024, 14336)
        c["K"] = _mult(rng, 2048, 14336, 256)
    elif kind == "train_dx":
        c["type"] = rng.choice(RECIPE)
        c["M"] = _log(rng, 128, 4096)
        c["N"] = _mult(rng, 1024, 14336, 32)
        c["K"] = _mult(rng, 2048, 5120, 256)
    elif kind == "moe":
        c["T"] = _log(rng, 1, 4096)
        c["E"] = rng.choice((16, 32, 64))
        c["topk"] = rng.choice((2, 4, 6, 8))
        c["hidden"] = _mult(rng, 1024, 2816, 256)
        c["ffn"] = _mult(rng, 512, 1536, 32)
    else:
        c["M"] = _log(rng, 128, 4096)
        c["N"] = _mult(rng, 1024, 14336, 8)
        c["K"] = _mult(rng, 1024, 14336, 32)
    if "M" in c and "N" in c:  # no dearer than the largest listed case
        most = 6.0e11 if kind == "train_dx" else 8.0e11
        while 2.0 * c["M"] * c["N"] * c["K"] > most:
            c["M"] = max(2, c["M"] * 3 // 4)
    return c


class State:
    """What the program holds: tensors, raw addresses and handles."""


def _moe_route(c, g):
    """Top-k routing of T tokens: pairs sorted by expert (host offsets, device tables)."""
    T, E, k = c["T"], c["E"], c["topk"]
    p = torch.softmax(torch.randn((T, E), generator=g, device=DEV), -1)
    w, e = torch.topk(p, k, -1)
    order = torch.argsort(e.reshape(-1), stable=True)
    place = torch.empty_like(order)
    place[order] = torch.arange(T * k, device=DEV)
    counts = torch.bincount(e.reshape(-1), minlength=E).tolist()
    off = [0]
    for n in counts:
        off.append(off[-1] + n)
    return off, place.to(torch.int32).view(T, k).contiguous(), w.reshape(-1)[order].contiguous()


def _operands(case, seed, values=False):
    """The tensors of a case, the same for prepare and exact: (weights, inputs, routing)."""
    c, g = case, _gen(seed)
    kind = c["kind"]
    if kind in ("gemv", "dense"):
        return [weight(c["type"], c["N"], c["K"], g, values)], [_x(g, c["K"])], None
    if kind == "layer":
        ws = [weight(t, N, K, g, values) for t, N, K in _layer(c)]
        return ws, {K: _x(g, c["M"], K) for K in sorted({K for _, _, K in _layer(c)})}, None
    if kind in ("prompt", "rows", "train_fwd"):
        return [weight(c["type"], c["N"], c["K"], g, values)], [_x(g, c["M"], c["K"])], None
    if kind == "train_dx":
        ws = [weight(c["type"], c["N"], c["K"], g, values) for _ in range(2)]
        return ws, [_x(g, c["M"], c["N"]) for _ in range(2)], None
    if kind == "moe":
        H, F, E = c["hidden"], c["ffn"], c["E"]
        ws = [weight("q4_K", E * 2 * F, H, g, values), weight("q5_0", E * H, F, g, values)]
        P = c["T"] * c["topk"]
        return ws, [_x(g, P, H), _x(g, P, F)], _moe_route(c, g)
    return [(_x(g, c["N"], c["K"]).mul_(0.02), None)], [_x(g, c["M"], c["K"])], None


def prepare(case, seed):
    s, c = State(), case
    ws, xs, route = _operands(c, seed)
    s.case, s.keep, s.w = c, xs, [w for w, _ in ws]
    kind = c["kind"]
    if kind in ("gemv", "dense"):
        s.y = _y(c["N"])
        s.args = (s.w[0].data_ptr(), TYPES[c["type"]], row_bytes(c["type"], c["K"]), xs[0].data_ptr(), s.y.data_ptr(),
                  c["N"], c["K"])
    elif kind == "layer":
        s.chat = tier_amd.Chat()
        s.y, s.calls = [], []
        for (t, N, K), w in zip(_layer(c), s.w):
            i = s.chat.add(TYPES[t], N, K, dev=w.data_ptr())
            y = _y(c["M"], N)
            s.y.append(y)
            s.calls.append((i, xs[K].data_ptr(), y.data_ptr(), c["M"]))
        s.chat.place()
    elif kind == "prompt":
        s.y = _y(c["M"], c["N"])
        t = TYPES[c["type"]]
        s.ws = _ws(tier_amd.qgemm_ws_bytes(t, c["M"], c["N"], c["K"], tier_amd.MODE_F32))
        s.args = (s.w[0].data_ptr(), t, row_bytes(c["type"], c["K"]), xs[0].data_ptr(), s.y.data_ptr(), c["M"], c["N"],
                  c["K"], s.ws.data_ptr(), s.ws.numel())
    elif kind == "rows":
        s.y = _y(c["M"], c["N"])
        s.ws = _ws(tier_amd.x3_rows_ws_bytes(c["M"], c["K"], c["N"]))
        s.call = tier_amd.chat_fp3 if c["type"] == "f16" else tier_amd.chat_bf3
        s.args = (s.w[0].data_ptr(), xs[0].data_ptr(), s.y.data_ptr(), c["M"], c["K"], c["N"], c["N"], s.ws.data_ptr(),
                  s.ws.numel())
    elif kind == "train_fwd":
        s.y = _y(c["M"], c["N"])
        t = TYPES[c["type"]]
        s.ws = _ws(tier_amd.qgemm_ws_bytes(t, c["M"], c["N"], c["K"], tier_amd.MODE_X3REF))
        s.args = (s.w[0].data_ptr(), t, row_bytes(c["type"], c["K"]), xs[0].data_ptr(), s.y.data_ptr(), c["M"], c["N"],
                  c["K"], c["N"], tier_amd.MODE_X3REF, 0.0, s.ws.data_ptr(), s.ws.numel())
    elif kind == "train_dx":
        s.y = _y(c["M"], c["K"])
        s.w16 = [torch.zeros((c["N"], c["K"]), dtype=torch.float16, device=DEV) for _ in range(2)]
        s.ws = _ws(tier_amd.x3_gemm_ws_bytes(c["K"], c["M"], c["N"]))
    elif kind == "moe":
        H, F, E, T, k = c["hidden"], c["ffn"], c["E"], c["T"], c["topk"]
        s.off, s.pairs, s.pw = route
        P = T * k
        s.gu, s.dn, s.out = _y(P, 2 * F), _y(P, H), _y(T, H)
        s.calls = []
        for w, t, N, K, x, y in ((s.w[0], "q4_K", 2 * F, H, xs[0], s.gu), (s.w[1], "q5_0", H, F, xs[1], s.dn)):
            rb = row_bytes(t, K)
            s.calls.append(([w.data_ptr() + e * N * rb for e in range(E)], [TYPES[t]] * E, [rb] * E, x.data_ptr(),
                            y.data_ptr(), N, K))
        s.ws = _ws(max(tier_amd.qgemm_grouped_ws_bytes(q, s.off, N, K) for _, q, _, _, _, N, K in s.calls))
    else:
        M, N, K = c["M"], c["N"], c["K"]
        half = lambda r: torch.zeros((r, K), dtype=torch.float16, device=DEV)  # noqa: E731
        s.parts = [half(M), half(M), half(N), half(N)]
        s.exps = [torch.zeros(r, dtype=torch.int32, device=DEV) for r in (M, N)]
        s.y = _y(M, N)
        tier_amd.x3s_split(s.w[0].data_ptr(), s.parts[2].data_ptr(), s.parts[3].data_ptr(), s.exps[1].data_ptr(), N, K)
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "gemv":
        tier_amd.gemv_q(*s.args)
        return s.y
    if kind == "dense":
        W, t, _, x, y, N, K = s.args
        tier_amd.gemv(W, t, x, y, N, K)
        return s.y
    if kind == "layer":
        for i, x, y, M in s.calls:
            s.chat.lin(i, x, y, M)
        return s.y
    if kind == "prompt":
        W, t, rb, x, y, M, N, K, ws, nws = s.args
        tier_amd.qlinear(W, t, rb, x, y, M, N, K, ws, nws)
        return s.y
    if kind == "rows":
        if not s.call(*s.args):
            raise RuntimeError("shape not handled")
        return s.y
    if kind == "train_fwd":
        tier_amd.qgemm(*s.args)
        return s.y
    if kind == "train_dx":
        c = s.case
        M, N, K, t = c["M"], c["N"], c["K"], c["type"]
        for j in range(2):
            tier_amd.dq_launch(s.w[j].data_ptr(), TYPES[t], row_bytes(t, K), K, 0, N, s.w16[j].data_ptr(),
                               tier_amd.OUT_F16)
            tier_amd.fp3gemm(tier_amd.OP_N, K, M, N, s.w16[j].data_ptr(), K, s.keep[j].data_ptr(), float(j),
                             s.y.data_ptr(), K, s.ws.data_ptr(), s.ws.numel())
        return {"dx": s.y, "w16": s.w16}
    if kind == "moe":
        for W, q, rb, x, y, N, K in s.calls:
            tier_amd.qgemm_grouped(W, q, rb, x, s.off, y, N, K, tier_amd.MODE_X3REF, s.ws.data_ptr(), s.ws.numel())
        c = s.case
        tier_amd.moe_combine(s.dn.data_ptr(), s.pairs.data_ptr(), s.pw.data_ptr(), s.out.data_ptr(), c["T"], c["topk"],
                             c["hidden"])
        return {"gate_up": s.gu, "down": s.dn, "out": s.out}
    M, N, K = s.case["M"], s.case["N"], s.case["K"]
    xh, xl, wh, wl = (p.data_ptr() for p in s.parts)
    xe, we = (e.data_ptr() for e in s.exps)
    tier_amd.x3s_split(s.keep[0].data_ptr(), xh, xl, xe, M, K)
    tier_amd.x3s_gemm(xh, xl, xe, wh, wl, we, s.y.data_ptr(), M, N, K)
    return s.y


def work(case):
    c, kind = case, case["kind"]
    if kind in ("gemv", "dense"):
        N, K = c["N"], c["K"]
        return {"bytes": N * row_bytes(c["type"], K) + 4 * (N + K), "flops": 2 * N * K}
    if kind == "layer":
        L, M = _layer(c), c["M"]
        return {"bytes": sum(N * row_bytes(t, K) + 4 * M * N for t, N, K in L)
                + 4 * M * sum({K for _, _, K in L}), "flops": sum(2 * M * N * K for _, N, K in L)}
    if kind == "moe":
        # experts that some token of the batch takes, as independent draws of topk of E
        H, F, E, T, k = c["hidden"], c["ffn"], c["E"], c["T"], c["topk"]
        used = E * (1 - (1 - k / E) ** T)
        P = T * k
        return {"bytes": used * (2 * F * row_bytes("q4_K", H) + H * row_bytes("q5_0", F))
                + 4 * (P * (H + 2 * F) + P * (F + H) + T * H), "flops": 2 * P * 3 * F * H}
    M, N, K = c["M"], c["N"], c["K"]
    if kind == "train_dx":
        return {"bytes": 2 * (N * row_bytes(c["type"], K) + 2 * N * K + 4 * M * N) + 4 * M * K, "flops": 4 * M * N * K}
    w = 4 * N * K if kind == "x3s" else N * row_bytes(c["type"], K)
    return {"bytes": w + 4 * M * (N + K), "flops": 2 * M * N * K}


def tolerance(case):
    # fp32 results: sums of fp32-accurate products, in any order (measured against 64 bits:
    # up to 2.5e-7 for the GEMVs, 8e-7 for the split products)
    return {"rel": 3e-6, "max": 5e-5}


def exact(case, seed):
    c, kind = case, case["kind"]
    ws, xs, route = _operands(c, seed, True)
    vs = [v for _, v in ws]
    if kind in ("gemv", "dense"):
        return (vs[0].double() @ xs[0].double())
    if kind == "layer":
        return [_mul64(xs[K], v) for (_, _, K), v in zip(_layer(c), vs)]
    if kind in ("prompt", "rows"):
        return _mul64(xs[0], vs[0])
    if kind == "train_fwd":  # the weight is rounded to fp16 by definition
        return _mul64(xs[0], vs[0].half())
    if kind == "train_dx":
        w16 = [v.half() for v in vs]
        dx = xs[0].double() @ w16[0].double() + xs[1].double() @ w16[1].double()
        return {"dx": dx, "w16": [w.double() for w in w16]}
    if kind == "moe":
        H, F, E, T, k = c["hidden"], c["ffn"], c["E"], c["T"], c["topk"]
        off, pairs, pw = route
        gu = torch.zeros((T * k, 2 * F), dtype=torch.float64, device=DEV)
        dn = torch.zeros((T * k, H), dtype=torch.float64, device=DEV)
        for e in range(E):
            r = slice(off[e], off[e + 1])
            gu[r] = _mul64(xs[0][r], vs[0].view(E, 2 * F, H)[e].half())
            dn[r] = _mul64(xs[1][r], vs[1].view(E, H, F)[e].half())
        p = pairs.long().view(-1)
        out = (dn[p] * pw[p].double()[:, None]).view(T, k, H).sum(1)
        return {"gate_up": gu, "down": dn, "out": out}
    return _mul64(xs[0], ws[0][0])
