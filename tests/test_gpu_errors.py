"""Error paths of the library on a device: an allocation that fails inside a call reports
WL_E_NOMEM (BackendError, as the reference's OutOfMemoryException surfaces from its engine,
src/Server.cs:756-761) and leaves the context usable; the next call gives the same bits as a
context that never failed. The failure is injected on the host (wl_debug_fail_alloc), so no
kernel sees a bad pointer. A layer whose matrices do not fit together is refused before a launch."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_common import blocks
from windlass_amd import BackendError, LayerDesc, ShapeError, Transformer
from windlass_amd._lib import check, load
from windlass_amd.backend import Context, GgmlType

pytestmark = pytest.mark.gpu


@pytest.fixture
def fresh():
    ctx = Context(0)
    yield ctx
    check(load().wl_debug_fail_alloc(0))
    ctx.close()


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def test_failed_weight_upload_leaves_the_context_usable(fresh):
    t, rows, cols = GgmlType.Q4_K, 64, 512
    data = blocks(t, rows, cols, seed=3)
    x = np.random.default_rng(1).standard_normal((2, cols), dtype=np.float32)
    w0 = fresh.upload(t, data, rows, cols)
    want = Transformer.MatMul(w0, x, 2)
    check(load().wl_debug_fail_alloc(2))  # the next upload succeeds, the one after fails
    w1 = fresh.upload(t, data, rows, cols)
    with pytest.raises(BackendError, match="cannot allocate"):
        fresh.upload(t, data, rows, cols)
    w2 = fresh.upload(t, data, rows, cols)
    for w in (w0, w1, w2):
        assert np.array_equal(_bits(Transformer.MatMul(w, x, 2)), _bits(want))
        w.free()


@pytest.mark.parametrize("T", [1, 40])
def test_failed_scratch_growth_leaves_the_context_usable(fresh, T):
    # T = 40 runs the GEMM, whose staging needs the context's scratch: the first call on a new
    # context grows it, and that growth is the allocation made to fail
    t, rows, cols = GgmlType.Q6_K, 256, 1024
    data = blocks(t, rows, cols, seed=5)
    x = np.random.default_rng(T).standard_normal((T, cols), dtype=np.float32)
    ref = Context(0)
    try:
        wr = ref.upload(t, data, rows, cols)
        want = Transformer.MatMul(wr, x, T)
        wr.free()
    finally:
        ref.close()
    w = fresh.upload(t, data, rows, cols)
    check(load().wl_debug_fail_alloc(1))
    with pytest.raises(BackendError, match="cannot allocate"):
        Transformer.MatMul(w, x, T)
    assert np.array_equal(_bits(Transformer.MatMul(w, x, T)), _bits(want))
    w.free()


@pytest.mark.parametrize("odd", ["attn_k", "attn_v", "ffn_up"])
@pytest.mark.parametrize("cols", [256, 768])
def test_layer_refuses_matrices_of_other_columns(fresh, odd, cols):
    # the matrices that share x run in one launch in prompts of both kernels (20 and 200 tokens) and in
    # batch steps, on either arithmetic
    E, H, KH, HD, FF = 512, 4, 2, 64, 768
    t = GgmlType.Q4_K
    mats = {"attn_q": (H * HD, E), "attn_k": (KH * HD, E), "attn_v": (KH * HD, E), "attn_output": (E, H * HD),
            "ffn_gate": (FF, E), "ffn_up": (FF, E), "ffn_down": (E, FF)}
    mats[odd] = (mats[odd][0], cols)
    w = {n: fresh.upload(t, blocks(t, r, c, seed=1), r, c) for n, (r, c) in mats.items()}
    norm, x = torch.ones(E, device="cuda"), torch.ones((200, E), device="cuda")
    K, V = (torch.zeros((200, KH * HD), dtype=torch.int16, device="cuda") for _ in range(2))
    d = LayerDesc()
    for n in mats:
        setattr(d, n, w[n].handle.value)
    d.d_attn_norm = d.d_ffn_norm = norm.data_ptr()
    d.embd, d.heads, d.kv_heads, d.head_dim, d.rope_dims = E, H, KH, HD, HD
    d.rope_base, d.rope_freq_scale, d.eps = 10000.0, 1.0, 1e-6
    P = lambda v: ctypes.c_void_p(v.data_ptr())  # noqa: E731
    L, h = load(), fresh.handle
    torch.cuda.synchronize()
    for T in (1, 8, 20, 200):
        with pytest.raises(ShapeError):
            check(L.wl_layer_dev(h, ctypes.byref(d), P(x), T, 0, P(K), P(V)))
    for mma in (False, True):
        fresh.FloatMma = mma
        for N in (1, 8, 12):
            at = (ctypes.c_int32 * N)(*range(N))
            with pytest.raises(ShapeError):
                check(L.wl_layer_batch_dev(h, ctypes.byref(d), P(x), N, at, at, N, 16, P(K), P(V)))
    fresh.sync()
    assert bool((x == 1).all()) and not K.any() and not V.any()
    for m in w.values():
        m.free()
