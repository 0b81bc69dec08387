"""MoeFfn of more than 8 tokens at once on the matrix cores (src/Transformer.cs:253-311): against the
float64 product of the decoded experts, and a token's bits independent of the tokens beside it."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from gpu_common import blocks
from windlass_amd._lib import check, load
from windlass_amd.backend import Context

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def upload(ctx, gt, dt, ne, embd, ff):
    g, u, d = blocks(gt, ne * ff, embd, seed=1), blocks(gt, ne * ff, embd, seed=2), blocks(dt, ne * embd, ff, seed=3)
    ws = [ctx.upload(t, b, r, c, experts=ne) for t, b, r, c in ((gt, g, ff, embd), (gt, u, ff, embd), (dt, d, embd, ff))]
    return ws, [oracle.decode(t, b, n).astype(np.float64) for t, b, n in
                ((gt, g, ne * ff * embd), (gt, u, ne * ff * embd), (dt, d, ne * embd * ff))]


def dev_moe(ctx, logits, k, ws, x):
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    l, dx = torch.from_numpy(logits).cuda(), torch.from_numpy(x).cuda()
    y = torch.empty_like(dx)
    torch.cuda.synchronize()
    check(load().wl_moe_ffn_dev(ctx.handle, P(l), k, 1, ws[0].handle, ws[1].handle, ws[2].handle, P(dx), len(x), P(y)))
    ctx.sync()
    return y.cpu().numpy()


def moe64(logits, k, dense, x, ne, embd, ff):
    g, u, d = dense[0].reshape(ne, ff, embd), dense[1].reshape(ne, ff, embd), dense[2].reshape(ne, embd, ff)
    out = np.zeros((len(x), embd))
    for t in range(len(x)):
        sel, w, _ = oracle.route(logits[t], k, True)
        for e, wt in zip(sel, w):
            a = g[e] @ x[t].astype(np.float64)
            out[t] += float(wt) * (d[e] @ (a / (1 + np.exp(-np.clip(a, -700, 700))) * (u[e] @ x[t])))
    return out


# tokens: just past one pass of 8, either side of 16, 32 and 64 pairs per expert (the token tiles)
# and a tile with one pair; experts with no token at all (128), every token on one expert (1 of 2)
@pytest.mark.parametrize("types", [(12, 12), (12, 14), (14, 14), (14, 12)])
@pytest.mark.parametrize("ne,k,embd,ff,T", [(128, 8, 512, 256, 9), (16, 4, 512, 256, 17), (8, 2, 768, 512, 65),
                                            (8, 2, 256, 256, 130), (4, 4, 256, 256, 33), (60, 4, 256, 768, 300)])
def test_many_tokens(ctx, types, ne, k, embd, ff, T):
    ws, dense = upload(ctx, *types, ne, embd, ff)
    rng = np.random.default_rng(ne + T)
    x = rng.standard_normal((T, embd), dtype=np.float32)
    x[1] *= 1e8  # each token's parts have a scale of their own; its output (about x^2) stays in fp32's range
    x[2] *= 1e-8
    x[3, ::7] *= 300
    logits = rng.standard_normal((T, ne), dtype=np.float32)
    got = dev_moe(ctx, logits, k, ws, x)
    n = min(T, 24)
    pick = sorted(set([0, 1, 2, 3, T - 1]) | set(rng.choice(T, n, replace=False).tolist()))
    want = moe64(logits[pick], k, dense, x[pick], ne, embd, ff)
    # each product is within 1e-5 of sum |w x|, a few times a random row's spread: the bar of
    # the fp32 experts, token by token
    for i, t in enumerate(pick):
        assert np.max(np.abs(got[t] - want[i])) <= 1e-4 * np.std(want[i]), t
    # alone with eight others, and in another order, a token has the same bits
    sub = np.array([0, T - 1, 3, 1, T // 2, 2, 5, 6, 7])
    again = dev_moe(ctx, logits[sub], k, ws, x[sub])
    assert np.array_equal(again.view(np.uint32), got[sub].view(np.uint32))
    for w in ws:
        w.free()


def test_one_expert_takes_every_token(ctx):
    # every token of three tiles on the same two of 64 experts; a token of zeros, one with a NaN
    ne, k, embd, ff, T = 64, 2, 512, 256, 150
    ws, dense = upload(ctx, 12, 14, ne, embd, ff)
    rng = np.random.default_rng(0)
    x = rng.standard_normal((T, embd), dtype=np.float32)
    x[4] = 0
    x[5, 300] = np.nan
    logits = np.zeros((T, ne), np.float32)
    logits[:, 63], logits[:, 7] = 5, 4
    got = dev_moe(ctx, logits, k, ws, x)
    pick = [0, 31, 32, 63, 64, T - 1]
    want = moe64(logits[pick], k, dense, x[pick], ne, embd, ff)
    for i, t in enumerate(pick):
        assert np.max(np.abs(got[t] - want[i])) <= 1e-4 * np.std(want[i])
    assert not got[4].any() and np.isnan(got[5]).all()
    for w in ws:
        w.free()


@pytest.mark.parametrize("T", [1024, 1025, 2100])
def test_prompts_past_one_pass(ctx, T):
    # 1,024 tokens a pass at most: one full pass, two of 513 and 512, three of 700
    ne, k, embd, ff = 8, 2, 256, 512
    ws, dense = upload(ctx, 12, 14, ne, embd, ff)
    rng = np.random.default_rng(T)
    x, logits = rng.standard_normal((T, embd), dtype=np.float32), rng.standard_normal((T, ne), dtype=np.float32)
    got = dev_moe(ctx, logits, k, ws, x)
    # every token, in sets of 100 of other places
    order = rng.permutation(T)
    for i in range(0, T, 100):
        sub = order[i:i + 100] if T - i >= 109 else order[-100:]
        assert np.array_equal(dev_moe(ctx, logits[sub], k, ws, x[sub]).view(np.uint32), got[sub].view(np.uint32))
    pick = [0, 512, 513, 699, 700, 1023, T - 1]
    want = moe64(logits[pick], k, dense, x[pick], ne, embd, ff)
    for i, t in enumerate(pick):
        assert np.max(np.abs(got[t] - want[i])) <= 1e-4 * np.std(want[i]), t
    for w in ws:
        w.free()


def test_nan_logits_stay_with_their_token(ctx):
    # a NaN logit makes every probability NaN: the first k experts with NaN weights (src/Transformer.cs:313-340)
    ne, k, embd, ff, T = 16, 4, 256, 256, 40
    ws, _ = upload(ctx, 14, 12, ne, embd, ff)
    rng = np.random.default_rng(3)
    x, logits = rng.standard_normal((T, embd), dtype=np.float32), rng.standard_normal((T, ne), dtype=np.float32)
    want = dev_moe(ctx, logits, k, ws, x)
    logits[7, 5], logits[39] = np.nan, np.inf
    got = dev_moe(ctx, logits, k, ws, x)
    rest = [t for t in range(T) if t not in (7, 39)]
    assert np.isnan(got[[7, 39]]).all() and np.array_equal(got[rest].view(np.uint32), want[rest].view(np.uint32))
    for w in ws:
        w.free()
