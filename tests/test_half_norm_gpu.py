"""A projection whose pieces the next norm sums (ntk_gemm_half_defer, ntk_half_norm_split) and the product over that norm's halves (ntk_gemm_half_normed), against the launches one by one."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu
VP, I, F, Z = C.c_void_p, C.c_int, C.c_float, C.c_size_t


class HalfDesc(C.Structure):
    _fields_ = [("W", VP * 3), ("Y", VP * 3), ("out", I * 3), ("n", I), ("X", VP), ("n_tokens", I), ("in_features", I), ("accumulate", I), ("row_max", VP), ("silu", I),
                ("workspace", VP), ("workspace_bytes", Z)]


def _bind():
    L = _lib.lib()
    P = C.POINTER(_lib.GemmPartials)
    L.ntk_gemm_half.argtypes = [VP, VP, VP, I, I, I, I, VP, VP, Z, VP]
    L.ntk_gemm_half_defer.argtypes = [VP, VP, VP, I, I, I, VP, VP, Z, P, VP]
    L.ntk_half_norm_takes.argtypes = [I, I, Z]
    L.ntk_half_norm_split.argtypes = [VP, P, VP, I, I, F, VP, Z, VP]
    L.ntk_rmsnorm.argtypes = [VP, VP, VP, I, I, F, VP]
    L.ntk_gemm_half_many.argtypes, L.ntk_gemm_half_normed.argtypes = [C.POINTER(HalfDesc), VP], [C.POINTER(HalfDesc), P, VP]
    return L


# tokens from one up, widths of less than a workgroup, of its 8 x 256, 512 and 1024 threads with and without remainder, of two turns; K whose product splits and one whose does not
@pytest.mark.parametrize("T,H,K", [(1, 64, 64), (3, 2048, 4096), (200, 4096, 4096), (17, 4160, 14336), (33, 8256, 1024), (5, 16384, 192), (130, 3072, 8192)])
def test_norm_over_deferred_pieces(T, H, K):
    L, g = _bind(), np.random.default_rng(T + H + K)
    h0, x = (2 * g.standard_normal((T, H))).astype(np.float32), g.standard_normal((T, K)).astype(np.float32)
    W = DB.from_numpy((g.standard_normal((H, K)) / np.sqrt(K)).astype(np.float16))
    nw = DB.from_numpy((1 + 0.2 * g.standard_normal(H)).astype(np.float32))
    outs = (96, 160)
    U = [DB.from_numpy((g.standard_normal((o, H)) / np.sqrt(H)).astype(np.float16)) for o in outs]
    xb, n = DB.from_numpy(x), 4 * T * (max(H, K) + 1) + 64 + 16 * T * H * 4
    a, b = DB.zeros(n), DB.zeros(n)

    def product(call, X, *left):
        d, ys = HalfDesc(), [DB.zeros(T * o * 4) for o in outs]
        for i, o in enumerate(outs):
            d.W[i], d.Y[i], d.out[i] = U[i].ptr, ys[i].ptr, o
        d.n, d.X, d.n_tokens, d.in_features, d.workspace, d.workspace_bytes = 2, X.ptr, T, H, b.ptr, n
        _lib.check(call(C.byref(d), *left, None), "product")
        return [y.numpy(np.float32) for y in ys]

    one, norm = DB.from_numpy(h0), DB.zeros(T * H * 4)
    _lib.check(L.ntk_gemm_half(one.ptr, W.ptr, xb.ptr, T, H, K, 1, None, a.ptr, n, None), "half")
    _lib.check(L.ntk_rmsnorm(norm.ptr, one.ptr, nw.ptr, T, H, 1e-5, None), "norm")
    want = product(L.ntk_gemm_half_many, norm)
    hid, p = DB.from_numpy(h0), _lib.GemmPartials()
    assert L.ntk_half_norm_takes(T, H, n) == 1
    _lib.check(L.ntk_gemm_half_defer(hid.ptr, W.ptr, xb.ptr, T, H, K, None, a.ptr, n, C.byref(p), None), "defer")
    assert p.n_tokens == T and p.rows[0] == H and p.y[0] == hid.ptr and (p.nsplit > 1) == bool(p.part[0])
    _lib.check(L.ntk_half_norm_split(hid.ptr, C.byref(p), nw.ptr, T, H, 1e-5, b.ptr, n, None), "norm_split")
    got = product(L.ntk_gemm_half_normed, xb, None)
    assert np.array_equal(hid.numpy(np.float32), one.numpy(np.float32))
    _lib.check(L.ntk_half_norm_split(hid.ptr, None, nw.ptr, T, H, 1e-5, b.ptr, n, None), "norm_split")
    again = product(L.ntk_gemm_half_normed, xb, None)
    left = _lib.GemmPartials()
    product(L.ntk_gemm_half_normed, xb, C.byref(left))
    if left.nsplit > 1:                                                     # the matrices' pieces side by side, in the order that their sums take
        at = left.part[0] - b.ptr
        pieces = b.numpy(np.uint8)[at:at + 4 * left.nsplit * T * sum(outs)].view(np.float32).reshape(left.nsplit, T, sum(outs))
        tot = pieces[0]
        for u in range(1, left.nsplit):
            tot = tot + pieces[u]
        assert np.array_equal(tot[:, :outs[0]].reshape(-1), got[0]) and np.array_equal(tot[:, outs[0]:].reshape(-1), got[1])
    for w, q, r in zip(want, got, again):
        # the rows' norms differ by their sums' order alone: at most 2^-24 sqrt(H) / 2 of a value and the halves' 2^-23, near 1e-6 of the results' size
        assert np.isfinite(q).all() and np.abs(q - w).max() <= 4e-6 * max(np.abs(w).max(), 1e-3)
        assert np.array_equal(q, r)


def test_what_a_norm_over_halves_refuses():
    L = _bind()
    assert [L.ntk_half_norm_takes(*a) for a in ((4, 4096, 4 * 4097 * 4 + 32), (4, 4096, 4 * 4097 * 4 - 64), (0, 4096, 1 << 20), (4, 4100, 1 << 20), (4, 16448, 1 << 20))] == [1, 0, 0, 0, 0]
    h, w, b = DB.zeros(4 * 4096 * 4), DB.zeros(4096 * 4), DB.zeros(1 << 20)
    p = _lib.GemmPartials()
    p.nseg, p.n_tokens, p.nsplit, p.rows[0], p.y[0] = 1, 4, 1, 2048, h.ptr
    assert L.ntk_half_norm_split(h.ptr, C.byref(p), w.ptr, 4, 4096, 1e-5, b.ptr, 1 << 20, None) != 0
    assert L.ntk_half_norm_split(h.ptr + 4, None, w.ptr, 4, 2048, 1e-5, b.ptr, 1 << 20, None) != 0
