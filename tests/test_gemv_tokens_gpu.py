"""ntk_gemv_tokens: the products of a prompt's tokens in one launch hold the bits of a launch a token."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib, gguf as G
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu
VP, I = C.c_void_p, C.c_int


@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("T,out,K", [(2, 1024, 1024), (4, 9, 8), (5, 7, 520), (16, 2048, 1024), (33, 256, 2048), (200, 65, 1032)])
def test_tokens_hold_the_bits_of_one(half, T, out, K):
    L, g = _lib.lib(), np.random.default_rng(T + out + K)
    L.ntk_gemv_tokens.argtypes = [VP, VP, VP, I, I, I, I, VP]
    L.ntk_gemv.argtypes = [VP, VP, VP, I, I, I, VP]
    dt = G.DT_F16 if half else G.DT_F32
    W = DB.from_numpy(g.standard_normal((out, K)).astype(np.float16 if half else np.float32))
    x, y, one = DB.from_numpy(g.standard_normal((T, K)).astype(np.float32)), DB.zeros(T * out * 4), DB.zeros(T * out * 4)
    _lib.check(L.ntk_gemv_tokens(y.ptr, W.ptr, x.ptr, T, out, K, dt, None), "tokens")
    for t in range(T):
        _lib.check(L.ntk_gemv(one.ptr + 4 * t * out, W.ptr, x.ptr + 4 * t * K, out, K, dt, None), "one")
    assert np.array_equal(y.numpy(np.float32), one.numpy(np.float32))


def test_what_the_tokens_refuse():
    L = _lib.lib()
    L.ntk_gemv_tokens.argtypes = [VP, VP, VP, I, I, I, I, VP]
    b = DB.zeros(1 << 16)
    for a in ((2, 4, 12, G.DT_F16), (2, 4, 16, G.DT_Q8_0), (-1, 4, 16, G.DT_F16)):
        assert L.ntk_gemv_tokens(b.ptr, b.ptr, b.ptr, *a, None) != 0


@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("add", [0, 1])
@pytest.mark.parametrize("rows,K", [((1024, 256, 256), 1024), ((3, 5), 72), ((9000,), 520), ((1, 0, 2), 9)])
def test_matrices_in_one_launch(half, add, rows, K):
    L, g = _lib.lib(), np.random.default_rng(sum(rows) + K)
    L.ntk_gemv_dense.argtypes = [C.POINTER(_lib.GemvSeg), I, VP, I, I, VP]
    L.ntk_gemv.argtypes = [VP, VP, VP, I, I, I, VP]
    dt = G.DT_F16 if half else G.DT_F32
    x = DB.from_numpy(g.standard_normal(K).astype(np.float32))
    W = [DB.from_numpy(g.standard_normal((max(r, 1), K)).astype(np.float16 if half else np.float32)) for r in rows]
    old = [g.standard_normal(max(r, 1)).astype(np.float32) for r in rows]
    y, one, segs = [DB.from_numpy(o) for o in old], [DB.zeros(4 * max(r, 1)) for r in rows], (_lib.GemvSeg * len(rows))()
    for i, r in enumerate(rows):
        segs[i].W, segs[i].y, segs[i].rows, segs[i].dtype = W[i].ptr, y[i].ptr, r, dt
        _lib.check(L.ntk_gemv(one[i].ptr, W[i].ptr, x.ptr, r, K, dt, None), "one")
    _lib.check(L.ntk_gemv_dense(segs, len(rows), x.ptr, K, add, None), "dense")
    for i, r in enumerate(rows):
        want = one[i].numpy(np.float32)[:r]
        assert np.array_equal(y[i].numpy(np.float32)[:r], old[i][:r] + want if add else want)
    segs[0].dtype = G.DT_Q8_0
    assert L.ntk_gemv_dense(segs, len(rows), x.ptr, K, add, None) != 0
