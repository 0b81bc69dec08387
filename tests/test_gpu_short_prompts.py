"""Prompts of 9 tokens and more over Q8_0, Q4_K, Q5_K, Q6_K and IQ4_XS rows. 9 to 128 tokens (Transformer.MatMul past 8 tokens, src/Transformer.cs:526-536) on the
kernel that reads and decodes each weight once for all tokens: at the edges of its 16-token tiles
and 16- and 32-row groups, with fewer column blocks than waves, and inside a layer, where the
matrices that share x run in one launch and the norm and the SiLU write the operands."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_common import GEMM_REL, bf16_round, blocks, decoded, tol_check
from windlass_amd import LayerDesc, Transformer
from windlass_amd._lib import check, load
from windlass_amd.backend import Context, GgmlType

pytestmark = pytest.mark.gpu
TYPES = [GgmlType.Q8_0, GgmlType.Q4_K, GgmlType.Q5_K, GgmlType.Q6_K, GgmlType.IQ4_XS]


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


# one block of columns and fewer than the four waves, an odd count (rows of 2-byte formats at both
# alignments); one row, a ragged last group, and enough rows for groups of 32 (8,200 on 256 CUs)
@pytest.mark.parametrize("t", TYPES, ids=lambda t: t.name)
@pytest.mark.parametrize("rows,cols", [(1, 256), (37, 1280), (8200, 768), (500, 4352)])
@pytest.mark.parametrize("T", [9, 16, 17, 48, 65, 113, 128])
def test_bars(ctx, t, rows, cols, T):
    data = blocks(t, rows, cols, seed=rows + cols + int(t))
    x = np.random.default_rng(T).standard_normal((T, cols), dtype=np.float32)
    w = ctx.upload(t, data, rows, cols)
    y = Transformer.MatMul(w, x, T)
    wd = decoded(t, data, rows, cols)
    # the bars of tests/test_gpu_gemm.py: fp32 accumulation of the bf16 operands, and bf16 itself
    tol_check(y, bf16_round(x), bf16_round(wd), rel=1e-5, what="bf16 operands")
    tol_check(y, x, wd, rel=GEMM_REL, what="fp32")
    w.free()


# rows past 10,240 columns, which eight waves share: an odd and an even count of column blocks, a ragged last
# group of 16 rows and of 32 (8,200 rows, where 101 of them are checked), beside 10,240 columns on four waves
@pytest.mark.parametrize("t", TYPES, ids=lambda t: t.name)
@pytest.mark.parametrize("rows,cols", [(37, 10240), (37, 10496), (20, 16384), (8200, 10496)])
def test_wide_bars(ctx, t, rows, cols):
    data = blocks(t, rows, cols, seed=rows + cols + int(t))
    w = ctx.upload(t, data, rows, cols)
    pick = np.arange(rows) if rows < 100 else np.r_[0:40, 4000:4021, rows - 40:rows]
    per = len(data) // rows
    wd = decoded(t, np.concatenate([data[r * per:r * per + per] for r in pick]), len(pick), cols)
    wb = bf16_round(wd)
    for T in (9, 17, 48, 64, 65, 96, 128):  # a kernel for each count of 16-token tiles
        x = np.random.default_rng(T).standard_normal((T, cols), dtype=np.float32)
        y = Transformer.MatMul(w, x, T)[:, pick]
        tol_check(y, bf16_round(x), wb, rel=1e-5, what="bf16 operands, T = %d" % T)
        tol_check(y, x, wd, rel=GEMM_REL, what="fp32, T = %d" % T)
    w.free()


# past 128 tokens: one more, the edges of 256- and 512-token tiles, K unsplit and split (one tile of
# 300 rows over 9 and 17 column blocks, 2,100 rows), a partly filled second tile
@pytest.mark.parametrize("t", TYPES, ids=lambda t: t.name)
@pytest.mark.parametrize("rows,cols,T", [(300, 2304, 129), (130, 256, 256), (300, 4352, 257), (2100, 512, 300),
                                         (129, 1024, 512), (257, 768, 530)])
def test_long_bars(ctx, t, rows, cols, T):
    test_bars(ctx, t, rows, cols, T)


def dev_rows(ctx, w, x, T, rows, pick):
    """Rows `pick` of W x for x [T][cols] in device memory."""
    y = torch.full((T, rows), float("nan"), device="cuda")
    torch.cuda.synchronize()
    check(load().wl_matmul_dev(ctx.handle, w.handle, -1, P(x), T, P(y)))
    ctx.sync()
    return y[pick].cpu().numpy()


# x of 2^31 values and a little more: its bf16 pieces pass 2 GiB at token 37,449 and 4 GiB at 74,898
def test_prompt_past_4_gib_of_pieces(ctx):
    rows, cols, T = 37, 28672, 75000
    x = torch.empty((T, cols), device="cuda")
    x.normal_(generator=torch.Generator(device="cuda").manual_seed(1))
    pick = [0, 37440, 37448, 37449, 60000, T - 150, T - 120, T - 1]
    xs = x[pick].cpu().numpy()
    for t in TYPES:
        data = blocks(t, rows, cols, seed=int(t))
        w = ctx.upload(t, data, rows, cols)
        tol_check(dev_rows(ctx, w, x, T, rows, pick), bf16_round(xs), bf16_round(decoded(t, data, rows, cols)), rel=1e-5,
                  what=t.name)
        w.free()


# one block of columns more than the long prompts' kernel takes: x zero but for the ends of the row
# and of the first half, so that the fp32 sums stay as short as elsewhere
def test_prompt_past_the_widest_rows(ctx):
    rows, cols, T = 3, (1 << 22) + 256, 129
    x = torch.zeros((T, cols), device="cuda")
    at = [slice(0, 512), slice(cols // 2 - 300, cols // 2 + 300), slice(cols - 512, cols)]
    g = torch.Generator(device="cuda").manual_seed(2)
    for a in at:
        x[:, a].normal_(generator=g)
    pick = [0, 31, 127, 128]
    part = lambda v: bf16_round(np.concatenate([v[:, a] for a in at], 1))  # noqa: E731
    xs = part(x[pick].cpu().numpy())
    for t in TYPES:
        data = blocks(t, rows, cols, seed=int(t))
        w = ctx.upload(t, data, rows, cols)
        tol_check(dev_rows(ctx, w, x, T, rows, pick), xs, part(decoded(t, data, rows, cols)), rel=1e-5, what=t.name)
        w.free()


def P(t):
    return ctypes.c_void_p(t.data_ptr())


# one order of x for q, k and v (one launch), two (one by one); down of either order
@pytest.mark.parametrize("qkv,gu,down", [(("Q4_K", "Q5_K", "Q6_K"), "Q4_K", "Q6_K"), (("Q8_0",) * 3, "IQ4_XS", "Q8_0"),
                                         (("Q4_K", "Q8_0", "Q6_K"), "Q6_K", "IQ4_XS")])
@pytest.mark.parametrize("T", [9, 47, 128, 200])
def test_layer_equals_its_operations(ctx, qkv, gu, down, T):
    layer_equals_its_operations(ctx, qkv, gu, down, T, 512)


# gate and up over rows that eight waves share
@pytest.mark.parametrize("qkv,gu,down", [(("Q4_K", "Q5_K", "Q6_K"), "Q4_K", "Q6_K"), (("Q8_0",) * 3, "IQ4_XS", "Q8_0"),
                                         (("Q6_K",) * 3, "Q6_K", "Q5_K"), (("Q8_0",) * 3, "Q8_0", "Q4_K")])
@pytest.mark.parametrize("T", [9, 31, 47, 61, 90, 128])
def test_wide_layer_equals_its_operations(ctx, qkv, gu, down, T):
    layer_equals_its_operations(ctx, qkv, gu, down, T, 10496)


def layer_equals_its_operations(ctx, qkv, gu, down, T, E):
    """A prompt's layer gives the bits of its operations called one at a time (past 128 tokens q, k and v
    may split K otherwise together than alone: the last bit of a sum moves, and some bf16 and fp16
    roundings with it)."""
    L, h, rng = load(), ctx.handle, np.random.default_rng(T)
    H, KH, HD, FF, pos0 = 4, 2, 64, 768, 3
    mats = {"attn_q": (qkv[0], H * HD, E), "attn_k": (qkv[1], KH * HD, E), "attn_v": (qkv[2], KH * HD, E),
            "attn_output": ("Q4_K", E, H * HD), "ffn_gate": (gu, FF, E), "ffn_up": (gu, FF, E), "ffn_down": (down, E, FF)}
    w = {n: ctx.upload(GgmlType[t], blocks(GgmlType[t], r, c, seed=i), r, c) for i, (n, (t, r, c)) in enumerate(mats.items())}
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    norms = [dev((1 + 0.1 * rng.standard_normal(E)).astype(np.float32)) for _ in range(2)]
    d = LayerDesc()
    for n in mats:
        setattr(d, n, w[n].handle.value)
    d.d_attn_norm, d.d_ffn_norm = (v.data_ptr() for v in norms)
    d.embd, d.heads, d.kv_heads, d.head_dim, d.rope_dims = E, H, KH, HD, HD
    d.rope_base, d.rope_freq_scale, d.eps, d.residual_scale = 10000.0, 1.0, 1e-6, 0.5
    x0 = rng.standard_normal((T, E), dtype=np.float32)
    cache = rng.standard_normal((pos0 + T, KH * HD)).astype(np.float16).view(np.int16)
    xa, Ka, Va, xb, Kb, Vb = dev(x0), dev(cache), dev(cache), dev(x0), dev(cache), dev(cache)
    xn, o = torch.empty((T, E), device="cuda"), torch.empty((T, E), device="cuda")
    q, k, v, att = (torch.empty((T, n), device="cuda") for n in (H * HD, KH * HD, KH * HD, H * HD))
    g, u = torch.empty((T, FF), device="cuda"), torch.empty((T, FF), device="cuda")
    f = ctypes.c_float
    torch.cuda.synchronize()
    check(L.wl_layer_dev(h, ctypes.byref(d), P(xa), T, pos0, P(Ka), P(Va)))
    mm = lambda n, x, y: check(L.wl_matmul_dev(h, w[n].handle, -1, P(x), T, P(y)))  # noqa: E731
    check(L.wl_rms_norm_dev(h, P(xb), T, E, P(norms[0]), f(1e-6), P(xn)))
    mm("attn_q", xn, q), mm("attn_k", xn, k), mm("attn_v", xn, v)
    for y, nh in ((q, H), (k, KH)):
        check(L.wl_rope_dev(h, P(y), T, nh, HD, HD, 0, pos0, None, 10000.0, 1.0, None))
    check(L.wl_kv_store_dev(h, P(k), P(v), T, KH * HD, P(Kb), P(Vb), pos0))
    check(L.wl_attention_dev(h, P(q), T, H, KH, HD, P(Kb), P(Vb), pos0, f(HD ** -0.5), P(att)))
    mm("attn_output", att, o)
    check(L.wl_residual_dev(h, P(xb), P(o), T * E, f(0.5)))
    check(L.wl_rms_norm_dev(h, P(xb), T, E, P(norms[1]), f(1e-6), P(xn)))
    mm("ffn_gate", xn, g), mm("ffn_up", xn, u)
    ctx.sync()
    gd = g.double()
    h32 = ((g / (1 + torch.exp(-gd).float())) * u).contiguous()  # SwiGlu's operations (src/Transformer.cs:247)
    torch.cuda.synchronize()
    mm("ffn_down", h32, o)
    check(L.wl_residual_dev(h, P(xb), P(o), T * E, f(0.5)))
    ctx.sync()
    if T <= 128:
        assert torch.equal(Ka, Kb) and torch.equal(Va, Vb)
    else:  # fp16 values one step apart at most
        for a, b in ((Ka, Kb), (Va, Vb)):
            a, b = a.view(torch.float16).float(), b.view(torch.float16).float()
            assert bool(((a - b).abs() <= 2.0 ** -10 * b.abs() + 2.0 ** -14).all())
    # h is rounded to bf16: a last-bit difference between the two exponentials moves few values by one step
    diff = (xa - xb).abs()
    assert (T > 128 or float((diff > 0).float().mean()) < 0.02) and float(diff.max()) <= 2.0 ** -8 * float(xb.abs().max())
    for m in w.values():
        m.free()
