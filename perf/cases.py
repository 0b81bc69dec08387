"""The work a user's program has this library do, as cases that can be timed and compared.

listed() names the calls one by one, draw() gives more of the same ranges. prepare() makes what the
program holds before the call (weights uploaded as raw GGUF blocks, activations, filled KV caches),
run() is one pass through the public entry points, and exact() is the same result in 64 bits from
plain torch, decoded here from the block layouts alone.

The kinds of call:
  host    Transformer.MatMul on host arrays, the engine's own seam
  matmul  wl_matmul_dev, one matrix on activations in device memory
  layer   an embedding and one decoder layer of one sequence: a decode step (T = 1) or a prompt
  batch   an embedding and one decoder layer for the next tokens of several sequences
  moe     the routed experts of one MoE layer, given the router's logits
  model   DeviceTransformer.forward_ids: embedding, layers, final norm and head; returns logits
"""
import ctypes
import math

import numpy as np
import torch

from windlass_amd import Transformer
from windlass_amd._lib import check, load
from windlass_amd.backend import Context, GgmlType, LayerDesc
from windlass_amd.model import DeviceTransformer, ModelConfig

EPS = 1e-5
ROPE_BASE = 500000.0
EMBD_ROWS = 1000  # rows of the embedding table the layer and batch cases read their tokens from

# decoder layers by size: embd, heads, kv heads, head dim, FFN (the 8B and 70B Llama layers of the
# benchmark, and the shape of a 1B model: head dim 64)
DIMS = {"1b": (2048, 32, 8, 64, 8192), "8b": (4096, 32, 8, 128, 14336), "70b": (8192, 64, 8, 128, 28672)}

# weight formats of a layer's attn_v and ffn_down, and of its other matrices
MIXES = {"q4_k_m": ("Q6_K", "Q4_K"), "q4_k": ("Q4_K", "Q4_K"), "q5_k_m": ("Q6_K", "Q5_K"), "q6_k": ("Q6_K", "Q6_K"),
         "q8_0": ("Q8_0", "Q8_0"), "iq4_xs": ("IQ4_XS", "IQ4_XS")}


def listed():
    return [
        # one product of a small model through the engine's seam: the smallest call, copies and all
        {"name": "host_q8_0_4096_t1", "kind": "host", "type": "Q8_0", "rows": 4096, "cols": 4096, "T": 1},
        # a 70B down projection in a format with a lookup table, at one token
        {"name": "iq4_xs_8192x28672_t1", "kind": "matmul", "type": "IQ4_XS", "rows": 8192, "cols": 28672, "T": 1},
        # a prompt of ordinary length through a format that is neither Q4_K nor Q6_K
        {"name": "q8_0_14336x4096_t200", "kind": "matmul", "type": "Q8_0", "rows": 14336, "cols": 4096, "T": 200},
        # a decode step of a small dense model with its head, the loop a chat user waits on
        {"name": "model_8b_2l_t1", "kind": "model", "dims": "8b", "mix": "q4_k_m", "layers": 2, "vocab": 128256,
         "T": 1, "pos0": 700},
        # a decode step of the headline's model late in a long conversation
        {"name": "layer_70b_t1_at_4000", "kind": "layer", "dims": "70b", "mix": "q4_k_m", "T": 1, "pos0": 4000},
        # a server's step: eight sequences of different lengths, the default arithmetic
        {"name": "batch_70b_8", "kind": "batch", "dims": "70b", "mix": "q4_k_m", "N": 8, "positions": 1000,
         "mode": "float"},
        # a larger step of a server that chose the matrix cores
        {"name": "batch_8b_16_mma", "kind": "batch", "dims": "8b", "mix": "q4_k_m", "N": 16, "positions": 500,
         "mode": "mma"},
        # a short question: most prompts of a chat
        {"name": "layer_8b_t45", "kind": "layer", "dims": "8b", "mix": "q4_k_m", "T": 45, "pos0": 300},
        # the prefill of the headline's model
        {"name": "layer_70b_t512", "kind": "layer", "dims": "70b", "mix": "q4_k_m", "T": 512, "pos0": 0},
        # the second part of a long document's prompt
        {"name": "layer_8b_t2048_at_2048", "kind": "layer", "dims": "8b", "mix": "q4_k_m", "T": 2048, "pos0": 2048},
        # a decode step of a 128-expert model's FFN
        {"name": "moe_t1", "kind": "moe", "embd": 2048, "ff": 768, "experts": 128, "used": 8, "gu": "Q4_K",
         "down": "Q4_K", "T": 1},
        # the same FFN in a prompt
        {"name": "moe_t300", "kind": "moe", "embd": 2048, "ff": 768, "experts": 128, "used": 8, "gu": "Q4_K",
         "down": "Q6_K", "T": 300},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "matmul", "matmul", "layer", "layer", "layer", "batch", "moe", "moe", "model"])
    if kind == "host":
        return {"kind": kind, "type": rng.choice(["Q8_0", "Q4_K", "Q6_K"]), "rows": _log(rng, 256, 16384),
                "cols": 256 * _log(rng, 2, 32), "T": rng.choice([1, 1, 1, 2, 7, _log(rng, 9, 128)])}
    if kind == "matmul":
        cols = 256 * _log(rng, 4, 112)
        return {"kind": kind, "type": rng.choice(["Q8_0", "Q4_K", "Q6_K", "Q5_K", "IQ4_XS"]),
                "rows": _log(rng, 512, min(28672, 28672 * 8192 // cols)), "cols": cols,
                "T": rng.choice([1, 1, rng.randint(2, 8), _log(rng, 9, 600), _log(rng, 9, 600)])}
    if kind == "layer":
        T = rng.choice([1, rng.randint(2, 8), _log(rng, 9, 128), _log(rng, 9, 128), _log(rng, 129, 1024)])
        dims = rng.choice(["1b", "8b", "8b", "70b"]) if T <= 256 else rng.choice(["1b", "8b"])
        return {"kind": kind, "dims": dims, "mix": rng.choice(["q4_k_m", "q4_k_m", "q5_k_m", "q8_0", "iq4_xs"]), "T": T,
                "pos0": rng.choice([0, _log(rng, 10, 3000)])}
    if kind == "batch":
        return {"kind": kind, "dims": rng.choice(["1b", "8b", "8b", "70b"]), "mix": rng.choice(["q4_k_m", "q4_k", "q6_k"]),
                "N": rng.randint(2, 20), "positions": _log(rng, 40, 2000), "mode": rng.choice(["float", "mma", "int"])}
    if kind == "moe":
        return {"kind": kind, "embd": rng.choice([1024, 2048]), "ff": rng.choice([512, 768, 1024, 1536]),
                "experts": rng.choice([8, 32, 60, 64, 128]), "used": rng.choice([2, 4, 6, 8]),
                "gu": rng.choice(["Q4_K", "Q4_K", "Q6_K"]), "down": rng.choice(["Q4_K", "Q6_K"]),
                "T": rng.choice([1, rng.randint(2, 8), _log(rng, 9, 300), _log(rng, 9, 300)])}
    return {"kind": kind, "dims": rng.choice(["1b", "8b"]), "mix": rng.choice(["q4_k_m", "q8_0"]), "layers": rng.randint(1, 3),
            "vocab": rng.choice([32000, 128256]), "T": rng.choice([1, 1, _log(rng, 9, 128)]), "pos0": _log(rng, 1, 3000)}


# ------------------------------------------------------------------ weights: raw blocks and values

# per format: values and bytes of a block
LAYOUT = {"Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210), "IQ4_XS": (256, 136)}
KVALUES = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000 + salt)
    return g


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _blocks(t, rows, cols, seed, salt, std=None):
    """rows x cols values of format t as raw blocks [nb][bytes] on the GPU: quants over their whole
    range, block scales that give the values the deviation of a trained layer, 1 / sqrt(cols)."""
    g = _gen(seed, salt)
    be, bb = LAYOUT[t]
    nb = rows * (cols // be)
    std = std or 1.0 / math.sqrt(cols)
    b = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, device="cuda", generator=g)
    spread = torch.rand(nb, device="cuda", generator=g) * 0.8 + 0.6
    if t == "Q8_0":
        b[:, :2] = _half_bytes(spread * (std / 73.6))
    elif t in ("Q4_K", "Q5_K"):
        top = 15 if t == "Q4_K" else 31
        sc = torch.randint(20, 64, (nb, 8), dtype=torch.int32, device="cuda", generator=g)
        # the sub-blocks' minimums equal their scales and dmin = d * top / 2: values centred on zero
        lo, hi = sc[:, :4], sc[:, 4:]
        b[:, 4:8] = (lo | (hi >> 4 << 6)).to(torch.uint8)
        b[:, 8:12] = (lo | (hi >> 4 << 6)).to(torch.uint8)
        b[:, 12:16] = ((hi & 15) | ((hi & 15) << 4)).to(torch.uint8)
        d = spread * (std / ((top + 1) / math.sqrt(12) * 42))
        b[:, 0:2] = _half_bytes(d)
        b[:, 2:4] = _half_bytes(d * (top / 2))
    elif t == "Q6_K":
        sc = torch.randint(32, 128, (nb, 16), dtype=torch.int32, device="cuda", generator=g)
        sign = torch.randint(0, 2, (nb, 16), dtype=torch.int32, device="cuda", generator=g) * 2 - 1
        b[:, 192:208] = (sc * sign).to(torch.int8).view(torch.uint8)
        b[:, 208:210] = _half_bytes(spread * (std / (18.5 * 84)))
    else:  # IQ4_XS
        b[:, :2] = _half_bytes(spread * (std / (67.0 * 18.5)))
    return b


def _values(t, b):
    """The values of raw blocks b [nb][bytes], in 64 bits."""
    nb = b.shape[0]
    half = lambda lo: b[:, lo:lo + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if t == "Q8_0":
        return half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    i = b.to(torch.int32)
    if t in ("Q4_K", "Q5_K"):
        s = i[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
        qs = i[:, _quants_at(t):].reshape(nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(nb, 8, 32)
        if t == "Q5_K":
            bit = torch.arange(8, device=b.device, dtype=torch.int32).reshape(1, 8, 1)
            q = q + ((i[:, None, 16:48] >> bit & 1) << 4)
        v = half(0)[:, :, None] * sc[:, :, None].double() * q.double() - half(2)[:, :, None] * mn[:, :, None].double()
        return v.reshape(nb, 256)
    if t == "Q6_K":
        ql, qh = i[:, :128].reshape(nb, 2, 2, 32), i[:, 128:192].reshape(nb, 2, 1, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        q = torch.cat([ql & 15, ql >> 4], 2)  # [nb][half][4 runs][32]
        shift = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int32).reshape(1, 1, 4, 1)
        q = (q | ((qh >> shift & 3) << 4)) - 32
        return (half(208)[:, :, None] * sc[:, :, None] * q.reshape(nb, 16, 16).double()).reshape(nb, 256)
    sh = i[:, 2:3] | (i[:, 3:4] << 8)  # IQ4_XS
    n = torch.arange(8, device=b.device, dtype=torch.int32)
    sl = i[:, 4:8].repeat_interleave(2, 1) >> (4 * (n & 1)) & 15
    ls = (sl | ((sh >> (2 * n) & 3) << 4)) - 32
    qs = i[:, 8:].reshape(nb, 8, 16)
    table = torch.tensor(KVALUES, dtype=torch.float64, device=b.device)
    q = table[torch.cat([qs & 15, qs >> 4], 2).long()]
    return (half(0)[:, :, None] * ls[:, :, None].double() * q).reshape(nb, 256)


def _quants_at(t):
    return 16 if t == "Q4_K" else 48


def _dense(t, rows, cols, seed, salt, std=None):
    """The matrix of _blocks in 64 bits [rows][cols]."""
    b = _blocks(t, rows, cols, seed, salt, std)
    out = torch.empty((b.shape[0], LAYOUT[t][0]), dtype=torch.float64, device="cuda")
    step = 1 << 17
    for i in range(0, b.shape[0], step):
        out[i:i + step] = _values(t, b[i:i + step])
    return out.reshape(rows, cols)


def _bytes(t, rows, cols):
    be, bb = LAYOUT[t]
    return rows * (cols // be) * bb


# ----------------------------------------------------------------------------------- the state

_contexts = {}


def _context(mode):
    """One context per arithmetic, as one program has one engine; every state of it shares its stream."""
    c = _contexts.get(mode)
    if c is None:
        c = _contexts[mode] = Context(0)
        c.FloatMma = mode == "mma"
        c.IntDot = mode == "int"
    return c


class State:
    """A case's buffers and weights; the weights go with it."""

    def __init__(self, case):
        self.case, self.ctx, self.weights = case, _context(case.get("mode", "float")), []

    def upload(self, t, rows, cols, seed, salt, experts=1, std=None):
        b = _blocks(t, rows * experts, cols, seed, salt, std).cpu().numpy()
        w = self.ctx.upload(GgmlType[t], b, rows, cols, experts)
        self.weights.append(w)
        return w

    def __del__(self):
        for w in getattr(self, "weights", []):
            w.free()


def _normal(shape, seed, salt, scale=1.0):
    return torch.randn(shape, device="cuda", generator=_gen(seed, salt)) * scale


def _cache(rows, kd, seed, salt):
    return _normal((rows, kd), seed, salt).to(torch.float16)


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


NAMES = ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")


def _shapes(dims, mix):
    """{tensor: (format, rows, cols)} of a layer."""
    E, H, KH, HD, F = DIMS[dims]
    odd, rest = MIXES[mix]
    size = {"attn_q": (H * HD, E), "attn_k": (KH * HD, E), "attn_v": (KH * HD, E), "attn_output": (E, H * HD),
            "ffn_gate": (F, E), "ffn_up": (F, E), "ffn_down": (E, F)}
    return {n: (odd if n in ("attn_v", "ffn_down") else rest,) + size[n] for n in NAMES}


def _norm_vector(n, seed, salt):
    return 1.0 + _normal((n,), seed, salt, 0.1)


def _layer_state(s, case, seed):
    """A layer's weights and description, its embedding table and the norm vectors."""
    E, H, KH, HD, F = DIMS[case["dims"]]
    d = LayerDesc()
    for i, (n, (t, rows, cols)) in enumerate(_shapes(case["dims"], case["mix"]).items()):
        setattr(d, n, s.upload(t, rows, cols, seed, i).handle.value)
    s.norms = [_norm_vector(E, seed, 20), _norm_vector(E, seed, 21)]
    d.d_attn_norm, d.d_ffn_norm = (v.data_ptr() for v in s.norms)
    d.embd, d.heads, d.kv_heads, d.head_dim, d.rope_dims = E, H, KH, HD, HD
    d.rope_base, d.rope_freq_scale, d.eps = ROPE_BASE, 1.0, EPS
    s.desc = d
    s.embd = s.upload("Q8_0", EMBD_ROWS, E, seed, 30, std=1.0)
    n = case["T"] if case["kind"] == "layer" else case["N"]
    s.ids = _ids(n, EMBD_ROWS, seed)
    s.x = torch.empty((n, E), device="cuda")


def _ids(n, vocab, seed):
    return torch.randint(0, vocab, (n,), dtype=torch.int32, device="cuda", generator=_gen(seed, 31))


def _batch_rows(case):
    """Position and slot of each row: lengths from short to full, slots in another order."""
    N, top = case["N"], case["positions"]
    pos = [top - 1 - (i * top) // N * (i % 3) // 2 for i in range(N)]
    return pos, [(5 * i + 3) % N if N % 5 else N - 1 - i for i in range(N)]


def _moe_logits(case, seed):
    return _normal((case["T"], case["experts"]), seed, 2)


def prepare(case, seed):
    s = State(case)
    kind = case["kind"]
    if kind in ("host", "matmul"):
        s.w = s.upload(case["type"], case["rows"], case["cols"], seed, 0)
        s.x = _normal((case["T"], case["cols"]), seed, 1)
        if kind == "host":
            s.x = s.x.cpu().numpy()
        else:
            s.y = torch.empty((case["T"], case["rows"]), device="cuda")
    elif kind == "layer":
        _layer_state(s, case, seed)
        E, H, KH, HD, F = DIMS[case["dims"]]
        p, T = case["pos0"], case["T"]
        s.K, s.V = _cache(p + T, KH * HD, seed, 40), _cache(p + T, KH * HD, seed, 41)
        s.out = {"x": s.x, "k": s.K[p:], "v": s.V[p:]}
    elif kind == "batch":
        _layer_state(s, case, seed)
        E, H, KH, HD, F = DIMS[case["dims"]]
        N, cap = case["N"], case["positions"]
        pos, slot = _batch_rows(case)
        s.pos, s.slot = (ctypes.c_int32 * N)(*pos), (ctypes.c_int32 * N)(*slot)
        s.K = _cache(N * cap, KH * HD, seed, 40).reshape(N, cap, KH * HD)
        s.V = _cache(N * cap, KH * HD, seed, 41).reshape(N, cap, KH * HD)
        s.out = {"x": s.x, "k": [s.K[b, a] for a, b in zip(pos, slot)], "v": [s.V[b, a] for a, b in zip(pos, slot)]}
    elif kind == "moe":
        E, F, n = case["embd"], case["ff"], case["experts"]
        s.gate = s.upload(case["gu"], F, E, seed, 0, experts=n)
        s.up = s.upload(case["gu"], F, E, seed, 1, experts=n)
        s.down = s.upload(case["down"], E, F, seed, 3, experts=n)
        s.logits = _moe_logits(case, seed)
        s.x = _normal((case["T"], E), seed, 4)
        s.y = torch.empty((case["T"], E), device="cuda")
    else:
        _model_state(s, case, seed)
    torch.cuda.synchronize()  # the context's stream does not wait for torch's
    return s


def _model_state(s, case, seed):
    E, H, KH, HD, F = DIMS[case["dims"]]
    odd = MIXES[case["mix"]][0]
    w = {"token_embd": s.upload("Q8_0", EMBD_ROWS, E, seed, 30, std=1.0),
         "output": s.upload(odd, case["vocab"], E, seed, 32)}
    v = {"output_norm": _norm_vector(E, seed, 22)}
    for l in range(case["layers"]):
        for i, (n, (t, rows, cols)) in enumerate(_shapes(case["dims"], case["mix"]).items()):
            w["blk.%d.%s" % (l, n)] = s.upload(t, rows, cols, seed, 100 * l + 100 + i)
        v["blk.%d.attn_norm" % l] = _norm_vector(E, seed, 100 * l + 120)
        v["blk.%d.ffn_norm" % l] = _norm_vector(E, seed, 100 * l + 121)
    cfg = ModelConfig(layers=case["layers"], embd=E, heads=H, kv_heads=KH, head_dim=HD, rope_base=ROPE_BASE, eps=EPS)
    p, T = case["pos0"], case["T"]
    m = s.model = DeviceTransformer(s.ctx, cfg, w, v, p + T)
    for l in range(case["layers"]):
        m.K[l].copy_(_cache(p + T, KH * HD, seed, 100 * l + 140).view(torch.int16))
        m.V[l].copy_(_cache(p + T, KH * HD, seed, 100 * l + 141).view(torch.int16))
    m.length = p
    s.ids = _ids(T, EMBD_ROWS, seed)
    s.out = {"logits": m.logits, "k": m.K.view(torch.float16)[:, p:], "v": m.V.view(torch.float16)[:, p:]}


def run(s):
    case, L, h = s.case, load(), s.ctx.handle
    kind = case["kind"]
    if kind == "host":
        return Transformer.MatMul(s.w, s.x, case["T"])
    if kind == "matmul":
        check(L.wl_matmul_dev(h, s.w.handle, -1, _p(s.x), case["T"], _p(s.y)))
        return s.y
    if kind == "moe":
        check(L.wl_moe_ffn_dev(h, _p(s.logits), case["used"], 1, s.gate.handle, s.up.handle,
                                            s.down.handle, _p(s.x), case["T"], _p(s.y)))
        return s.y
    if kind == "model":
        s.model.forward_ids(s.ids, case["pos0"])
        return s.out
    check(L.wl_embed_dev_ids(h, s.embd.handle, _p(s.ids), s.x.shape[0], _p(s.x)))
    if kind == "layer":
        check(L.wl_layer_dev(h, ctypes.byref(s.desc), _p(s.x), case["T"], case["pos0"], _p(s.K), _p(s.V)))
    else:
        check(L.wl_layer_batch_dev(h, ctypes.byref(s.desc), _p(s.x), case["N"], s.pos, s.slot, case["N"],
                                                case["positions"], _p(s.K), _p(s.V)))
    return s.out


# ------------------------------------------------------------------------------- work, tolerance


def _layer_work(case, lengths, rows):
    """Bytes and operations of one layer for `rows` rows that attend to `lengths` positions each, the
    caches of distinct sequences read once (one sequence: the longest row's)."""
    E, H, KH, HD, F = DIMS[case["dims"]]
    sh = _shapes(case["dims"], case["mix"])
    kv = 2 * 2 * KH * HD * (max(lengths) if case["kind"] != "batch" else sum(lengths))
    return (sum(_bytes(*v) for v in sh.values()) + kv + 8 * rows * E,
            2 * rows * sum(r * c for _, r, c in sh.values()) + 4 * H * HD * sum(lengths))


def work(case):
    kind = case["kind"]
    if kind in ("host", "matmul"):
        r, c, T = case["rows"], case["cols"], case["T"]
        return {"bytes": _bytes(case["type"], r, c) + 4 * T * (r + c), "flops": 2 * T * r * c}
    if kind == "batch":
        b, f = _layer_work(case, [p + 1 for p in _batch_rows(case)[0]], case["N"])
        return {"bytes": b, "flops": f}
    if kind == "moe":
        E, F, n, k, T = case["embd"], case["ff"], case["experts"], case["used"], case["T"]
        distinct = n * (1 - (1 - k / n) ** T)
        one = 2 * _bytes(case["gu"], F, E) + _bytes(case["down"], E, F)
        return {"bytes": distinct * one + 4 * T * (n + 2 * E), "flops": 2 * T * k * 3 * E * F}
    T, p = case["T"], case["pos0"]
    b, f = _layer_work(case, [p + i + 1 for i in range(T)], T)
    if kind == "model":
        E = DIMS[case["dims"]][0]
        b = case["layers"] * b + _bytes(MIXES[case["mix"]][0], case["vocab"], E) + 4 * case["vocab"]
        f = case["layers"] * f + 2 * case["vocab"] * E
    return {"bytes": b, "flops": f}


def tolerance(case):
    """32-bit products up to 8 tokens (and the experts), bf16 operands past them, 8-bit activations
    under the integer switch. Layers return the fp16 rows of the caches too, where a change of the
    last 32-bit place moves some values by one fp16 step."""
    kind = case["kind"]
    if case.get("mode") == "int":
        return {"rel": 0.02, "max": 0.3}
    if kind == "moe":
        return {"rel": 4e-6, "max": 1e-4}
    if kind != "batch" and case["T"] > 8:
        return {"rel": 0.01, "max": 0.1}
    if kind in ("host", "matmul"):
        return {"rel": 4e-6, "max": 1e-4}
    return {"rel": 2e-4, "max": 4e-3}


# ----------------------------------------------------------------------------------- 64 bits


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, heads, hd, pos):
    i = torch.arange(hd // 2, dtype=torch.float64, device="cuda")
    a = pos.double()[:, None] * ROPE_BASE ** (-2 * i / hd)
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    v = x.reshape(-1, heads, hd // 2, 2)
    return torch.stack([v[..., 0] * c - v[..., 1] * s, v[..., 0] * s + v[..., 1] * c], -1).reshape(x.shape)


def _attention(q, K, V, heads, kv, hd, first):
    """q [T][heads * hd], caches [n][kv * hd]: row t attends to positions 0 .. first + t."""
    T, n, out = q.shape[0], K.shape[0], torch.empty_like(q)
    dead = torch.arange(n, device="cuda")[None] > first + torch.arange(T, device="cuda")[:, None]
    for h in range(heads):
        a, b = slice(h * hd, h * hd + hd), h // (heads // kv) * hd
        s = q[:, a] @ K[:, b:b + hd].double().t() / math.sqrt(hd)
        out[:, a] = torch.softmax(s.masked_fill(dead, -math.inf), 1) @ V[:, b:b + hd].double()
    return out


def _exact_layer(case, x, seed, salt, norms, attend):
    """One layer of x; attend(q, k, v) stores the rows' keys and values and returns the attention."""
    mat = {}
    for i, (n, (t, rows, cols)) in enumerate(_shapes(case["dims"], case["mix"]).items()):
        mat[n] = (lambda a, t=t, rows=rows, cols=cols, i=i: a @ _dense(t, rows, cols, seed, salt + i).t())
    a = _rms(x, norms[0])
    x = x + mat["attn_output"](attend(mat["attn_q"](a), mat["attn_k"](a), mat["attn_v"](a)))
    a = _rms(x, norms[1])
    g = mat["ffn_gate"](a)
    return x + mat["ffn_down"](g * torch.sigmoid(g) * mat["ffn_up"](a))


def _attend_one(case, K, V, kept):
    """attend() of one sequence whose rows start at pos0 of the caches K, V (fp16, written); kept
    takes the new keys and values before they are rounded to fp16."""
    E, H, KH, HD, F = DIMS[case["dims"]]
    p, T = case["pos0"], case["T"]
    pos = torch.arange(p, p + T, device="cuda")

    def attend(q, k, v):
        k = _rope(k, KH, HD, pos)
        kept.append((k, v))
        K[p:p + T], V[p:p + T] = k.half(), v.half()
        return _attention(_rope(q, H, HD, pos), K, V, H, KH, HD, p)
    return attend


def exact(case, seed):
    """run()'s result in 64 bits. The attention reads the caches' fp16 values; the new cache rows are
    given before their rounding to fp16, whose steps a 32-bit difference can move either way."""
    kind = case["kind"]
    if kind in ("host", "matmul"):
        x = _normal((case["T"], case["cols"]), seed, 1).double()
        y = x @ _dense(case["type"], case["rows"], case["cols"], seed, 0).t()
        return y.cpu().numpy() if kind == "host" else y
    if kind == "moe":
        return _exact_moe(case, seed)
    E, H, KH, HD, F = DIMS[case["dims"]]
    table = _dense("Q8_0", EMBD_ROWS, E, seed, 30, std=1.0)
    if kind == "batch":
        N, cap = case["N"], case["positions"]
        K, V = _cache(N * cap, KH * HD, seed, 40).reshape(N, cap, -1), _cache(N * cap, KH * HD, seed, 41).reshape(N, cap, -1)
        pos, slot = _batch_rows(case)
        at, kept = torch.tensor(pos, device="cuda"), []

        def attend(q, k, v):
            q, k, out = _rope(q, H, HD, at), _rope(k, KH, HD, at), torch.empty_like(q)
            kept.append((k, v))
            for i, (a, b) in enumerate(zip(pos, slot)):
                K[b, a], V[b, a] = k[i].half(), v[i].half()
                out[i:i + 1] = _attention(q[i:i + 1], K[b, :a + 1], V[b, :a + 1], H, KH, HD, a)
            return out
        x = _exact_layer(case, table[_ids(N, EMBD_ROWS, seed).long()], seed, 0,
                         [_norm_vector(E, seed, 20), _norm_vector(E, seed, 21)], attend)
        return {"x": x, "k": list(kept[0][0]), "v": list(kept[0][1])}
    p, T = case["pos0"], case["T"]
    x = table[_ids(T, EMBD_ROWS, seed).long()]
    kept = []
    for l in range(case.get("layers", 1)):
        s = 100 * l + 100 if kind == "model" else 0
        K, V = _cache(p + T, KH * HD, seed, s + 40), _cache(p + T, KH * HD, seed, s + 41)
        x = _exact_layer(case, x, seed, s, [_norm_vector(E, seed, s + 20), _norm_vector(E, seed, s + 21)],
                         _attend_one(case, K, V, kept))
    if kind == "layer":
        return {"x": x, "k": kept[0][0], "v": kept[0][1]}
    lg = _rms(x[-1:], _norm_vector(E, seed, 22)) @ _dense(MIXES[case["mix"]][0], case["vocab"], E, seed, 32).t()
    return {"logits": lg, "k": torch.stack([k for k, _ in kept]),
            "v": torch.stack([v for _, v in kept])}


def _exact_moe(case, seed):
    E, F, n, k, T = case["embd"], case["ff"], case["experts"], case["used"], case["T"]
    prob = torch.softmax(_moe_logits(case, seed).double(), 1)
    top, sel = torch.topk(prob, k, 1)
    top = top / top.sum(1, keepdim=True)
    x = _normal((T, E), seed, 4).double()
    gate = _dense(case["gu"], n * F, E, seed, 0).reshape(n, F, E)
    up = _dense(case["gu"], n * F, E, seed, 1).reshape(n, F, E)
    down = _dense(case["down"], n * E, F, seed, 3).reshape(n, E, F)
    out = torch.zeros((T, E), dtype=torch.float64, device="cuda")
    for e in range(n):
        t, j = torch.nonzero(sel == e, as_tuple=True)
        if t.numel():
            g = x[t] @ gate[e].t()
            out[t] += top[t, j][:, None] * ((g * torch.sigmoid(g) * (x[t] @ up[e].t())) @ down[e].t())
    return out
