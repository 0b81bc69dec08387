"""Attention of a prompt's rows on the matrix cores (16 rows and more; Attention,
src/Transformer.cs:351-393) against float64, at the edges of its 32-token blocks, 64-position steps and
position chunks, with infinities and NaN in the caches, and against the row-by-row kernels' error."""
import ctypes
import math

import numpy as np
import pytest
import torch

from windlass_amd._lib import check, load
from windlass_amd.backend import Context

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def run(ctx, q, K, V, heads, kvh, hd, pos0, scale, rows=None):
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    T = q.shape[0]
    out = torch.full((T, heads * hd), 7.0, device="cuda")
    step = rows or T
    torch.cuda.synchronize()
    for t0 in range(0, T, step):
        n = min(step, T - t0)
        check(load().wl_attention_dev(ctx.handle, P(q[t0:t0 + n]), n, heads, kvh, hd, P(K), P(V), pos0 + t0,
                                      ctypes.c_float(scale), P(out[t0:t0 + n])))
    ctx.sync()
    return out.double()


def ref(q, K, V, heads, kvh, hd, pos0, scale):
    T, n = q.shape[0], K.shape[0]
    out = torch.empty((T, heads * hd), dtype=torch.float64, device="cuda")
    dead = torch.arange(n, device="cuda")[None] > pos0 + torch.arange(T, device="cuda")[:, None]
    for h in range(heads):
        a, b = slice(h * hd, h * hd + hd), h // (heads // kvh) * hd
        s = (q[:, a].double() @ K[:, b:b + hd].double().t().contiguous()) * float(np.float32(scale))
        out[:, a] = torch.softmax(s.masked_fill(dead, -math.inf), 1) @ V[:, b:b + hd].double()
    return out


def case(T, heads, kvh, hd, pos0, qs=1.0, seed=0, extra=3):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed + T)
    n = pos0 + T
    q = torch.randn((T, heads * hd), device="cuda", generator=g) * qs
    K, V = (torch.randn((n + extra, kvh * hd), device="cuda", generator=g).half() for _ in range(2))
    K[n:], V[n:] = math.nan, math.nan  # past the last position: never read into a result
    return q, K, V, n


# one and two token blocks, a partial one; rows of exactly one step of 64 positions and one more;
# KV groups of 1, 2, 3, 4 and 8 heads (units past the last); chunks (few rows after many positions)
@pytest.mark.parametrize("heads,kvh,hd", [(4, 4, 64), (4, 2, 128), (6, 2, 128), (8, 2, 64), (16, 2, 128), (64, 8, 128)])
@pytest.mark.parametrize("T,pos0", [(16, 0), (32, 32), (33, 31), (64, 0), (65, 700), (130, 1)])
def test_against_float64(ctx, heads, kvh, hd, T, pos0):
    scale = 1 / math.sqrt(hd)
    q, K, V, n = case(T, heads, kvh, hd, pos0)
    got, want = run(ctx, q, K, V, heads, kvh, hd, pos0, scale), ref(q, K[:n], V[:n], heads, kvh, hd, pos0, scale)
    # the bar of every attention kernel: 2e-6 of the row's largest value
    err = (got - want).abs().max(1).values
    assert bool((err <= 2e-6 * want.abs().max(1).values).all()), err.max()


@pytest.mark.parametrize("qs,scale", [(1.0, 0.088), (30.0, 0.088), (1e-3, 1.0), (1e6, 1e-6), (1.0, -0.1), (1.0, 0.0)])
def test_error_no_larger_than_row_by_row(ctx, qs, scale):
    # wide and flat softmaxes, scaled queries, a negative and a zero scale: the root mean square
    # error against float64 next to the same rows in passes of 8 (the VALU kernel)
    heads, kvh, hd, T, pos0 = 8, 2, 128, 96, 2000
    q, K, V, n = case(T, heads, kvh, hd, pos0, qs, seed=5)
    want = ref(q, K[:n], V[:n], heads, kvh, hd, pos0, scale)
    rms = lambda y: float(((y - want) ** 2).mean().sqrt() / (want ** 2).mean().sqrt())  # noqa: E731
    new, old = rms(run(ctx, q, K, V, heads, kvh, hd, pos0, scale)), rms(run(ctx, q, K, V, heads, kvh, hd, pos0, scale, 8))
    print("rms error: tiles %.3g, rows %.3g" % (new, old))
    # a flat softmax (scale 0) is within two roundings of a fp32 result either way: 2^-23
    assert new <= max(1.05 * old, 2.0 ** -23)


# short prompts and flat softmaxes, where an error of the probabilities is not averaged over many terms
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("T,pos0", [(16, 0), (38, 0), (109, 0), (130, 300), (751, 1847)])
@pytest.mark.parametrize("qs", [0.1, 0.3, 1.0])
def test_error_no_larger_on_flat_softmaxes(ctx, qs, T, pos0, hd):
    heads, kvh, scale = 16, 4, hd ** -0.5
    q, K, V, n = case(T, heads, kvh, hd, pos0, qs, seed=17)
    want = ref(q, K[:n], V[:n], heads, kvh, hd, pos0, scale)
    rms = lambda y: float(((y - want) ** 2).mean().sqrt() / (want ** 2).mean().sqrt())  # noqa: E731
    new, old = rms(run(ctx, q, K, V, heads, kvh, hd, pos0, scale)), rms(run(ctx, q, K, V, heads, kvh, hd, pos0, scale, 8))
    print("rms error: tiles %.3g, rows %.3g" % (new, old))
    assert new <= 1.05 * old


@pytest.mark.parametrize("qs", [1e9, 1e13, 1e30])
def test_scores_past_fp32_integers(ctx, qs):
    # scores whose last place in fp32 is many units: one key takes each row's whole weight
    heads, kvh, hd, T, pos0 = 4, 2, 64, 40, 300
    q, K, V, n = case(T, heads, kvh, hd, pos0, qs, seed=3)
    got, want = run(ctx, q, K, V, heads, kvh, hd, pos0, 0.125), ref(q, K[:n], V[:n], heads, kvh, hd, pos0, 0.125)
    assert float((got - want).abs().max()) <= 2e-6 * float(want.abs().max())


def test_nonfinite_rows_reach_only_their_readers(ctx):
    heads, kvh, hd, T, pos0 = 4, 2, 128, 70, 40
    q, K, V, n = case(T, heads, kvh, hd, pos0, seed=9)
    K[60, 5], V[75, 3], V[90, 130], K[100, 200] = math.inf, -math.inf, math.nan, math.nan
    got, old = run(ctx, q, K, V, heads, kvh, hd, pos0, 0.088), run(ctx, q, K, V, heads, kvh, hd, pos0, 0.088, 8)
    same = got.isnan() == old.isnan()
    assert bool(same.all()) and bool((got.isinf() == old.isinf()).all())
    fin = old.isfinite()
    assert float((got - old)[fin].abs().max()) <= 4e-6 * float(old[fin].abs().max())


def test_many_heads_of_one_kv_head(ctx):
    # more than 65,535 groups of four (token block, head): 516 token blocks of 512 heads
    heads, hd, T = 512, 64, 16500
    g = torch.Generator(device="cuda").manual_seed(1)
    q, out = torch.empty((T, heads * hd), device="cuda").normal_(generator=g), torch.empty((T, heads * hd), device="cuda")
    K, V = (torch.randn((T, hd), device="cuda", generator=g).half() for _ in range(2))
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    torch.cuda.synchronize()
    check(load().wl_attention_dev(ctx.handle, P(q), T, heads, 1, hd, P(K), P(V), 0, ctypes.c_float(0.125), P(out)))
    ctx.sync()
    for t in (0, 31, 32, 8191, T - 1):
        got, qt, v = out[t].reshape(heads, hd).double(), q[t].reshape(heads, hd).double(), V[:t + 1].double()
        p = torch.softmax(qt @ K[:t + 1].double().t().contiguous() * 0.125, 1)
        # sixteen roundings of 2^-24 of the sum's size, sum p |v|: thousands of values nearly cancel here
        worst = float(((got - p @ v).abs() / (p @ v.abs())).max())
        assert worst <= 2.0 ** -20, (t, worst)
