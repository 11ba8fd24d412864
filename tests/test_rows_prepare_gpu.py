"""The producers of a long prompt's FP16 planes, four tokens a workgroup (ntk_rows_*_prepare_x): the workspace holds the bits that the launches of a token a workgroup leave."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib, ops
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu
VP, I, F = C.c_void_p, C.c_int, C.c_float


def _bind():
    L = _lib.lib()
    L.ntk_gemm_quant_workspace_bytes.restype = C.c_size_t
    L.ntk_rows_prepare_x.argtypes = L.ntk_gemm_prepare_x.argtypes = [VP, I, I, VP, VP]
    L.ntk_rows_norm_prepare_x.argtypes = [VP, C.POINTER(_lib.GemmPartials), VP, I, I, F, VP, VP, VP]
    L.ntk_rows_silu_mul_prepare_x.argtypes = [VP, C.POINTER(_lib.GemmPartials), VP, VP]
    return L


def _planes(L, T, W, fill, *, x=None):
    """the workspace's planes, sums and 1 / s after `fill`, or after the token-a-workgroup launch over x"""
    ws = DB.zeros(L.ntk_gemm_quant_workspace_bytes(W, 16))
    _lib.check(L.ntk_gemm_prepare_x(x.ptr, T, W, ws.ptr, None) if x is not None else fill(ws), "prepare")
    chunk = ((W // 32 + 1) * 8192 + (W // 32 + 15) // 8 * 2048 + 255) // 256 * 256
    return ws.numpy(np.uint8)[: 16 * chunk + 4 * ((T + 63) // 64 * 64)]


# tokens: the first of the range, remainders of a workgroup's four, of a record's sixteen and of a chunk, the largest; widths: less than a turn of the waves, whole and ragged turns
@pytest.mark.parametrize("T,W", [(65, 32), (66, 4096), (127, 160), (128, 2048), (131, 4128), (1003, 4096), (1024, 1056), (69, 8192), (70, 14336), (67, 12320)])
def test_planes_as_they_lie_and_of_a_gated_unit(T, W):
    L, g = _bind(), np.random.default_rng(T + W)
    x = (g.standard_normal((T, W)) * np.exp(g.standard_normal((T, 1)) * 4)).astype(np.float32)
    x[T // 2] = 0.0
    xb = DB.from_numpy(x)
    want = _planes(L, T, W, None, x=xb)
    assert np.array_equal(want, _planes(L, T, W, lambda ws: L.ntk_rows_prepare_x(xb.ptr, T, W, ws.ptr, None)))
    for nsplit in (1, 3):
        a, b = (DB.from_numpy(g.standard_normal((nsplit, T, W)).astype(np.float32)) for _ in range(2))
        p = _lib.GemmPartials()
        p.nseg, p.n_tokens, p.nsplit = 2, T, nsplit
        for i, q in enumerate((a, b)):
            p.rows[i], p.part[i], p.y[i] = W, q.ptr if nsplit > 1 else None, q.ptr
        out = DB.zeros(T * W * 4)
        got = _planes(L, T, W, lambda ws: L.ntk_rows_silu_mul_prepare_x(out.ptr, C.byref(p), ws.ptr, None))
        sa, sb = a.numpy(np.float32).reshape(nsplit, T, W).sum(0, dtype=np.float64), b.numpy(np.float32).reshape(nsplit, T, W).sum(0, dtype=np.float64)
        ref = sa / (1 + np.exp(-sa)) * sb
        o = out.numpy(np.float32).reshape(T, W)
        assert np.abs(o - ref).max() <= 2e-6 * np.abs(ref).max()            # (two sums of three, an exponential, a division and a product: eight roundings of 2^-24 at most, near 1e-6)
        assert np.array_equal(got, _planes(L, T, W, None, x=out))
        assert np.array_equal(got, _planes(L, T, W, lambda ws: L.ntk_rows_silu_mul_prepare_x(None, C.byref(p), ws.ptr, None)))


@pytest.mark.parametrize("T,H,nsplit", [(65, 64, 0), (1003, 4096, 2), (70, 4128, 1), (129, 8192, 4), (200, 2560, 8), (1024, 1024, 0)])
def test_planes_of_a_norm(T, H, nsplit):
    L, g = _bind(), np.random.default_rng(T + H)
    h0, w = (3 * g.standard_normal((T, H))).astype(np.float32), (1 + 0.2 * g.standard_normal(H)).astype(np.float32)
    parts = g.standard_normal((max(nsplit, 1), T, H)).astype(np.float32)
    hid, pb, wb, out = DB.from_numpy(h0), DB.from_numpy(parts), DB.from_numpy(w), DB.zeros(T * H * 4)
    p = _lib.GemmPartials()
    p.nseg, p.n_tokens, p.nsplit, p.rows[0], p.y[0], p.part[0] = 1, T, max(nsplit, 1), H, pb.ptr, pb.ptr if nsplit > 1 else None
    q = C.byref(p) if nsplit else None
    got = _planes(L, T, H, lambda ws: L.ntk_rows_norm_prepare_x(hid.ptr, q, wb.ptr, T, H, 1e-5, out.ptr, ws.ptr, None))
    want = h0
    if nsplit:
        want = parts[0]
        for s in range(1, nsplit):
            want = want + parts[s]
        want = want + h0
    assert np.array_equal(hid.numpy(np.float32).reshape(T, H), want)
    r = want.astype(np.float64)
    r = r / np.sqrt((r * r).mean(1, keepdims=True) + 1e-5) * w
    assert np.abs(out.numpy(np.float32).reshape(T, H) - r).max() <= 1e-6 * np.abs(r).max()      # (sums of at most 2^-24 sqrt(8192) / 2, halved by the root, and four roundings)
    assert np.array_equal(got, _planes(L, T, H, None, x=out))


def test_what_the_planes_of_four_tokens_refuse():
    L = _bind()
    L.ntk_rows_prepare_takes.argtypes = [I, I, I]
    assert [L.ntk_rows_prepare_takes(*a) for a in ((65, 8192, 1), (1024, 14336, 0), (64, 4096, 0), (1025, 4096, 0), (65, 8224, 1), (65, 14368, 0), (65, 4100, 0))] == [1, 1, 0, 0, 0, 0, 0]
    x, ws = DB.zeros(65 * 14368 * 4), DB.zeros(L.ntk_gemm_quant_workspace_bytes(14368, 16))
    assert L.ntk_rows_prepare_x(x.ptr, 65, 14368, ws.ptr, None) != 0 and L.ntk_rows_prepare_x(x.ptr + 4, 65, 4096, ws.ptr, None) != 0


def test_a_norm_clears_the_tokens_that_it_is_given():
    L, T, H = _bind(), 70, 256
    L.ntk_rows_norm_prepare_zero.argtypes = [VP, C.POINTER(_lib.GemmPartials), VP, I, I, F, VP, VP, VP, VP]
    hid, w, ws = DB.from_numpy(np.ones((T, H), np.float32)), DB.from_numpy(np.ones(H, np.float32)), DB.zeros(L.ntk_gemm_quant_workspace_bytes(H, 16))
    z = DB.from_numpy(np.full(T + 2, 3.0, np.float32))
    _lib.check(L.ntk_rows_norm_prepare_zero(hid.ptr, None, w.ptr, T, H, 1e-5, None, z.ptr, ws.ptr, None), "zero")
    assert np.array_equal(z.numpy(np.float32), np.r_[np.zeros(T), 3.0, 3.0].astype(np.float32))


def test_the_launch_is_taken_only_where_it_pays():
    """against the launch that leaves the rows with their maxima and the GEMM's own split, both in front of a product of 16 rows: a sixth in hand for the clock"""
    import time
    L = _bind()
    L.ntk_rows_prepare_pays.argtypes = [I, I, I, I]
    L.ntk_reduce_rmsnorm_rowmax.argtypes = [VP, C.POINTER(_lib.GemmPartials), VP, F, VP, VP, VP, VP]
    L.ntk_reduce_silu_mul_rowmax.argtypes = [VP, C.POINTER(_lib.GemmPartials), VP, VP]
    pays = L.ntk_rows_prepare_pays
    assert not pays(64, 4096, 0, 0) and not pays(100, 4096, 1, 8) and not pays(100, 4096, 1, 2) and not pays(100, 14336, 0, 1) and pays(100, 4096, 0, 0) and pays(1000, 4096, 1, 2) and pays(1000, 14336, 0, 1)
    most = 1024 * 14336 * 4
    hid, x, w, rm, W, y, a, b = (DB.zeros(n) for n in (most, most, 14336 * 4, 4096 * 4, 16 * 17 * 14336 // 16, 1024 * 64, 2 * most, 2 * most))
    ws = DB.zeros(L.ntk_gemm_quant_workspace_bytes(14336, 64))
    segs = (_lib.GemvSeg * 1)()
    segs[0].W, segs[0].y, segs[0].rows, segs[0].dtype = W.ptr, y.ptr, 16, 2
    for T, width, norm, nsplit in [(330, 4096, 1, 1), (600, 4096, 1, 2), (1000, 8192, 1, 2), (600, 2048, 1, 2), (700, 5632, 0, 1), (512, 14336, 0, 1), (700, 3072, 0, 2), (1000, 14336, 0, 2)]:
        assert pays(T, width, norm, nsplit)
        p = _lib.GemmPartials()
        p.nseg, p.n_tokens, p.nsplit = 1 if norm else 2, T, nsplit
        for i, q in enumerate((a, b)[:p.nseg]):
            p.rows[i], p.part[i], p.y[i] = width, q.ptr if nsplit > 1 else None, q.ptr

        def product(reuse):
            d = _lib.GemmDesc()
            d.segs, d.nseg, d.X, d.n_tokens, d.in_features, d.workspace, d.workspace_bytes, d.reuse_x, d.row_max = segs, 1, x.ptr, T, width, ws.ptr, ws.nbytes, reuse, None if reuse else rm.ptr
            _lib.check(L.ntk_gemm_quant_f16(C.byref(d), None), "product")

        def one():
            _lib.check(L.ntk_rows_norm_prepare_x(hid.ptr, C.byref(p), w.ptr, T, width, 1e-5, None, ws.ptr, None) if norm else L.ntk_rows_silu_mul_prepare_x(None, C.byref(p), ws.ptr, None), "one")
            product(1)

        def two():
            _lib.check(L.ntk_reduce_rmsnorm_rowmax(hid.ptr, C.byref(p), w.ptr, 1e-5, x.ptr, rm.ptr, None, None) if norm else L.ntk_reduce_silu_mul_rowmax(x.ptr, C.byref(p), rm.ptr, None), "two")
            product(0)
        best = {}
        for f in 5 * (one, two):
            L.ntk_stream_synchronize(None)
            t0 = time.perf_counter()
            for _ in range(60):
                f()
            L.ntk_stream_synchronize(None)
            best[f] = min(best.get(f, 1e9), time.perf_counter() - t0)
        print(T, width, norm, nsplit, "one %.1f two %.1f us" % (best[one] / 60e-6, best[two] / 60e-6))
        assert best[one] < 7 / 6 * best[two]
