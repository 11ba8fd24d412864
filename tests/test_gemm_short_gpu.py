"""Short prompts' projections over planes that their producers scale per token and 256 columns (ntk_short_*_prepare_x, ntk_gemm_short), against float64 products of the oracle's dequantised
weights: one block of 16 tokens and two, single tokens and whole blocks, rows that end inside a wave's 512 columns or inside a group, groups of very different size, one slice and several.

Tolerance, of the root of the sum of the products' squares: four times the 1.1e-6 that the oracle's own float32 products show on such matrices (2304 inputs; Q8_0 3.8e-7, Q4_K 6.1e-7, Q6_K
1.1e-6: sums in any order)."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib
from ntransformer_amd import gguf
from ntransformer_amd import gguf as G
from ntransformer_amd.ops import DeviceBuffer as DB
from oracle import arbiter
from oracle import oracle as O

pytestmark = pytest.mark.gpu
REL = 4.4e-6
VP = C.c_void_p


def lib():
    L = _lib.lib()
    L.ntk_gemm_quant_workspace_bytes.restype = C.c_size_t
    L.ntk_gemm_quant_workspace_bytes.argtypes = [C.c_int, C.c_int]
    L.ntk_gemm_short_takes.argtypes = [C.POINTER(C.c_int)] + [C.c_int] * 4
    L.ntk_short_prepare_x.argtypes = [VP, C.c_int, C.c_int, VP, VP]
    L.ntk_short_norm_prepare_x.argtypes = [VP, C.POINTER(_lib.GemmPartials), VP, C.c_int, C.c_int, VP, VP]
    L.ntk_short_silu_mul_prepare_x.argtypes = [C.POINTER(_lib.GemmPartials), VP, VP]
    L.ntk_gemm_short.argtypes = [C.POINTER(_lib.GemmDesc), C.c_int, C.c_float, C.c_size_t, VP]
    return L


def product(L, ws, nbytes, weights, ys, rows, dt, T, inf, normed=0, eps=0.0, resid=None, partials=None, part_at=0):
    segs = (_lib.GemvSeg * len(weights))()
    for i, (w, y) in enumerate(zip(weights, ys)):
        segs[i].W, segs[i].y, segs[i].rows, segs[i].dtype = w.ptr, y.ptr, rows, dt
    d = _lib.GemmDesc()
    d.segs, d.nseg, d.n_tokens, d.in_features, d.resid = segs, len(weights), T, inf, None if resid is None else resid.ptr
    d.workspace, d.workspace_bytes = ws.ptr, nbytes
    d.partials = C.pointer(partials) if partials is not None else None
    _lib.check(L.ntk_gemm_short(C.byref(d), normed, eps, part_at, None), "gemm_short")


def weights(r, gt, rows, inf):
    raw = np.frombuffer(G.synth_tensor(r, gt, rows, inf), np.uint8)
    dt = G.GGML_TO_DT[gt]
    return raw, arbiter.dequant(raw, rows, inf, dt).astype(np.float64).reshape(rows, inf), dt


def close(got, W, X):
    """got [T, rows] against W . X, by the products' sizes"""
    want = X @ W.T
    size = np.sqrt((X ** 2) @ (W ** 2).T)
    assert np.isfinite(got).all()
    assert (np.abs(got - want) <= REL * size + 1e-30).all(), float((np.abs(got - want) / (size + 1e-30)).max())


@pytest.mark.parametrize("qname", ["Q8_0", "Q4_0", "Q4_K", "Q5_K", "Q6_K"])
@pytest.mark.parametrize("T,rows,inf", [(1, 16, 256), (2, 48, 768), (16, 256, 1280), (17, 128, 512), (32, 64, 2304), (5, 2064, 256)])
def test_products_of_grouped_planes(qname, T, rows, inf):
    gt = getattr(G, "GGML_" + qname)
    L, r = lib(), np.random.Generator(np.random.Philox(key=[T, rows + inf]))
    dims = [(rows, inf)] + ([(rows, inf + 128)] if qname == "Q8_0" else [])      # Q8_0: a last group of half the columns, too
    for rows, inf in dims:
        one, two = (C.c_int * 1)(rows), (C.c_int * 2)(rows, rows)
        raw, W, dt = weights(r, gt, rows, inf)
        if not (L.ntk_gemm_short_takes(one, 1, max(T, 2), inf, dt) and L.ntk_gemm_short_takes(two, 2, max(T, 2), inf, dt)):
            assert qname == "Q6_K" and T > 16                                     # (32 tokens of the format that scales per 16 columns)
            continue
        Wd = DB.from_numpy(raw)
        nbytes = L.ntk_gemm_quant_workspace_bytes(inf, 2 * rows)
        ws, ws2 = DB(nbytes), DB(nbytes)
        X = r.standard_normal((T, inf)).astype(np.float32)
        X[:, 64:320] *= np.float32(1e4)                                           # groups of different sizes, zeros, one tiny and one huge row
        X[T // 2, : inf // 2] = 0.0
        X[0] *= np.float32(1e12)
        X[T - 1] *= np.float32(1e-12)
        y, Xd = DB.from_numpy(np.full((T, rows), 7.0, np.float32)), DB.from_numpy(X)
        _lib.check(L.ntk_short_prepare_x(Xd.ptr, T, inf, ws.ptr, None), "short_prepare_x")
        product(L, ws, nbytes, [Wd], [y], rows, dt, T, inf)
        close(y.numpy(np.float32).reshape(T, rows).astype(np.float64), W, X.astype(np.float64))
        # RMSNorm in front, a residual behind
        eps, nw = 1e-5, (1.0 + 0.1 * r.standard_normal(inf)).astype(np.float32)
        res = r.standard_normal((T, rows)).astype(np.float32)
        hd, nd = DB.from_numpy(X), DB.from_numpy(nw)
        _lib.check(L.ntk_short_norm_prepare_x(hd.ptr, None, nd.ptr, T, inf, ws.ptr, None), "short_norm")
        y = DB.from_numpy(res)
        product(L, ws, nbytes, [Wd], [y], rows, dt, T, inf, 1, eps, y)
        assert np.array_equal(hd.numpy(np.float32).reshape(T, inf), X)
        x64 = X.astype(np.float64)
        n64 = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + eps) * nw
        got = y.numpy(np.float32).reshape(T, rows).astype(np.float64)
        size = np.sqrt((n64 ** 2) @ (W ** 2).T) + np.abs(res)
        assert (np.abs(got - (res + n64 @ W.T)) <= REL * size).all()
        # sums of a gate | up launch -> silu * up -> sums of the next product -> its norm
        if rows % (128 if qname == "Q8_0" else 256) or not L.ntk_gemm_short_takes((C.c_int * 1)(rows), 1, max(T, 2), rows, dt):
            continue
        pt = _lib.GemmPartials()
        small = np.float32(1e-3) * r.standard_normal((T, inf)).astype(np.float32)
        xd = DB.from_numpy(small)
        _lib.check(L.ntk_short_prepare_x(xd.ptr, T, inf, ws.ptr, None), "short_prepare_x")
        g, u = DB.zeros(T * rows * 4), DB.zeros(T * rows * 4)
        product(L, ws, nbytes, [Wd, Wd], [g, u], rows, dt, T, inf, partials=pt)
        raw2, W2, _ = weights(r, gt, rows, rows)
        nb2 = L.ntk_gemm_quant_workspace_bytes(rows, 2 * rows)
        wa, wb, Wd2 = DB(nb2), DB(nb2), DB.from_numpy(raw2)
        _lib.check(L.ntk_short_silu_mul_prepare_x(C.byref(pt), wa.ptr, None), "short_silu")
        h0 = r.standard_normal((T, rows)).astype(np.float32)
        hd = DB.from_numpy(h0)
        pt2 = _lib.GemmPartials()
        product(L, wa, nb2, [Wd2], [hd], rows, dt, T, rows, resid=hd, partials=pt2)
        nw = (1.0 + 0.1 * r.standard_normal(rows)).astype(np.float32)
        nd = DB.from_numpy(nw)
        _lib.check(L.ntk_short_norm_prepare_x(hd.ptr, C.byref(pt2), nd.ptr, T, rows, wb.ptr, None), "short_norm")
        gv = small.astype(np.float64) @ W.T
        a = gv / (1.0 + np.exp(-gv)) * gv
        got = hd.numpy(np.float32).reshape(T, rows).astype(np.float64)
        # (the unit's own rounding beside the product's: gate and up carry REL of their sums' sizes each)
        ga = np.sqrt((small.astype(np.float64) ** 2) @ (W ** 2).T)
        ua = np.abs(gv) + ga
        size = np.sqrt((a ** 2) @ (W2 ** 2).T) + np.sqrt((2 * ga * ua) ** 2 @ (W2 ** 2).T) + np.abs(h0)
        assert (np.abs(got - (h0 + a @ W2.T)) <= REL * size).all()
        y = DB.zeros(T * rows * 4)
        product(L, wb, nb2, [Wd2], [y], rows, dt, T, rows, 1, eps)
        n64 = got / np.sqrt((got ** 2).mean(1, keepdims=True) + eps) * nw
        close(y.numpy(np.float32).reshape(T, rows).astype(np.float64), W2, n64)


def test_sums_side_by_side_and_what_is_refused():
    """two launches of different formats leave their sums in one workspace; shapes and sizes that the form does not take launch nothing"""
    L, r = lib(), np.random.Generator(np.random.Philox(key=[3, 9]))
    T, rows, inf = 16, 256, 2048
    raws = [np.frombuffer(G.synth_tensor(r, gt, rows, inf), np.uint8) for gt in (G.GGML_Q4_K, G.GGML_Q6_K)]
    dts = [G.GGML_TO_DT[gt] for gt in (G.GGML_Q4_K, G.GGML_Q6_K)]
    X = r.standard_normal((T, inf)).astype(np.float32)
    nbytes = L.ntk_gemm_quant_workspace_bytes(inf, 2 * rows)
    ws, Xd = DB(nbytes), DB.from_numpy(X)
    _lib.check(L.ntk_short_prepare_x(Xd.ptr, T, inf, ws.ptr, None), "short_prepare_x")
    bufs, sums, at = [DB.from_numpy(a) for a in raws], [], 0
    pts, ys = [_lib.GemmPartials(), _lib.GemmPartials()], [DB.zeros(T * rows * 4) for _ in dts]
    for w, y, dt, pt in zip(bufs, ys, dts, pts):
        product(L, ws, nbytes, [w], [y], rows, dt, T, inf, partials=pt, part_at=at)
        assert pt.nsplit > 1
        at += pt.nsplit * T * rows
    assert pts[1].part[0] - pts[0].part[0] == pts[0].nsplit * T * rows * 4
    ones, ws2 = DB.from_numpy(np.ones(rows, np.float32)), DB(nbytes)
    for raw, dt, pt in zip(raws, dts, pts):
        h = DB.zeros(T * rows * 4)
        _lib.check(L.ntk_short_norm_prepare_x(h.ptr, C.byref(pt), ones.ptr, T, rows, ws2.ptr, None), "short_norm")
        want = np.stack([O.gemv(raw, x, rows, inf, dt) for x in X]).astype(np.float64)
        got = h.numpy(np.float32).reshape(T, rows)
        assert np.abs(got - want).max() <= REL * 8 * np.abs(want).max()
    one = (C.c_int * 1)(rows)
    dt = dts[0]
    assert not L.ntk_gemm_short_takes(one, 1, 33, inf, dt) and not L.ntk_gemm_short_takes(one, 1, 16, inf + 32, dt)
    assert not L.ntk_gemm_short_takes((C.c_int * 1)(24), 1, 16, inf, dt) and not L.ntk_gemm_short_takes(one, 1, 16, inf, 0)
    assert L.ntk_short_prepare_x(ws.ptr, 33, inf, ws.ptr, None) != 0 and L.ntk_short_prepare_x(ws.ptr, 4, 40, ws.ptr, None) != 0


@pytest.mark.parametrize("T,H,G,splits,interleaved", [(1, 2, 1, (1, 1, 1), 0), (3, 6, 2, (4, 4, 17), 0), (16, 32, 8, (4, 4, 16), 0), (17, 4, 4, (2, 9, 10), 1), (32, 8, 1, (3, 1, 2), 0), (29, 64, 8, (8, 8, 8), 1)])
def test_attention_and_planes_in_one_launch(T, H, G, splits, interleaved):
    """against the three launches it replaces: the caches and the products of its planes bit for bit"""
    L, hd, rows = lib(), 128, 64
    g = np.random.default_rng(T + H)
    out = (H * hd, G * hd, G * hd)
    parts = [g.standard_normal((n, T, r)).astype(np.float32) for n, r in zip(splits, out)]
    parts[2][:, T // 2] *= np.float32(1e3)
    raw = np.frombuffer(gguf.synth_tensor(g, gguf.GGML_Q4_K, rows, H * hd), np.uint8)
    dt = gguf.GGML_TO_DT[gguf.GGML_Q4_K]
    L.ntk_short_angles.argtypes = [VP, C.c_int, C.c_float, C.c_float, VP]
    angles = DB.zeros(2 * 32 * hd // 2 * 4)
    _lib.check(L.ntk_short_angles(angles.ptr, hd, 500000.0, 1.0, None), "short_angles")
    nbytes = L.ntk_gemm_quant_workspace_bytes(H * hd, rows)
    L.ntk_reduce_rope_kv_store.argtypes = [VP, C.POINTER(VP), C.POINTER(C.c_int), VP] + [C.c_int] * 4 + [C.c_float, C.c_float, C.c_int, VP, VP, C.c_int, C.c_int, VP]
    L.ntk_attention_prefill.argtypes = [VP] * 4 + [C.c_int] * 6 + [C.c_float, VP]
    L.ntk_short_attention.argtypes = [C.POINTER(VP), C.POINTER(C.c_int), VP] + [C.c_int] * 4 + [C.c_float, C.c_int, VP, VP, C.c_int, VP, VP]
    scale, res = 1.0 / np.sqrt(np.float32(hd)), []
    for fused in (0, 1):
        kc, vc = (DB.from_numpy(np.full((T + 2, out[1]), 3.0, np.float16)) for _ in range(2))
        bufs, Wd = [DB.from_numpy(p) for p in parts], DB.from_numpy(raw)
        arr, ns, ws = (VP * 3)(*[b.ptr for b in bufs]), (C.c_int * 3)(*splits), DB(nbytes)
        if fused:
            _lib.check(L.ntk_short_attention(arr, ns, angles.ptr, T, H, G, hd, scale, interleaved, kc.ptr, vc.ptr, T + 2, ws.ptr, None), "short_attention")
        else:
            q, o, pos = DB.zeros(T * out[0] * 4), DB.zeros(T * out[0] * 4), DB.from_numpy(np.arange(T, dtype=np.int32))
            _lib.check(L.ntk_reduce_rope_kv_store(q.ptr, arr, ns, pos.ptr, T, H, G, hd, 500000.0, 1.0, interleaved, kc.ptr, vc.ptr, 0, T + 2, None), "rope")
            _lib.check(L.ntk_attention_prefill(o.ptr, q.ptr, kc.ptr, vc.ptr, T, 0, H, G, hd, T + 2, scale, None), "attention")
            _lib.check(L.ntk_short_prepare_x(o.ptr, T, H * hd, ws.ptr, None), "prepare")
        y = DB.zeros(T * rows * 4)
        product(L, ws, nbytes, [Wd], [y], rows, dt, T, H * hd)
        res.append((kc.numpy(np.uint16), vc.numpy(np.uint16), y.numpy(np.float32)))
    assert np.isfinite(res[0][2]).all()
    for a, b in zip(*res):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    assert L.ntk_short_attention(arr, ns, angles.ptr, 33, H, G, hd, scale, 0, kc.ptr, vc.ptr, 64, ws.ptr, None) != 0
    assert L.ntk_short_attention(arr, ns, angles.ptr, T, H + 1, 1, hd, scale, 0, kc.ptr, vc.ptr, T + 2, ws.ptr, None) != 0


@pytest.mark.parametrize("qname", ["Q8_0", "Q4_K", "Q6_K"])
@pytest.mark.parametrize("outliers", [0, 1])
@pytest.mark.parametrize("rows", [512, 16384])
def test_a_scale_per_group_is_no_further_from_64_bits_than_one_per_token(qname, outliers, rows):
    """the products of 16 tokens, 4096 inputs in many slices and in few: planes of a scale per token and 256 columns, whose sums are rounded once per unit, beside planes of one scale a token
    (ntk_gemm_quant_f16 over X), whose sums run on.  Root mean square of the error over the products' sizes; normal values, and five channels a thousand times as large.  0.53 to 1.0006 of it seen;
    the bound is 1.1: 16 x 512 products give either figure to within 2 %"""
    L, r = lib(), np.random.Generator(np.random.Philox(key=[11, outliers]))
    T, inf = 16, 4096
    raw, W, dt = weights(r, getattr(G, "GGML_" + qname), rows, inf)
    X = r.standard_normal((T, inf)).astype(np.float32)
    if outliers:
        X[:, [5, 1033, 2500, 3333, 4000]] *= np.float32(1e3)
    nbytes = L.ntk_gemm_quant_workspace_bytes(inf, rows)
    ws, Wd, Xd = DB(nbytes), DB.from_numpy(raw), DB.from_numpy(X)
    want = X.astype(np.float64) @ W.T
    size = np.sqrt((X.astype(np.float64) ** 2) @ (W ** 2).T)
    errs = []
    for short in (1, 0):
        y = DB.zeros(T * rows * 4)
        if short:
            _lib.check(L.ntk_short_prepare_x(Xd.ptr, T, inf, ws.ptr, None), "short_prepare_x")
            product(L, ws, nbytes, [Wd], [y], rows, dt, T, inf)
        else:
            segs = (_lib.GemvSeg * 1)()
            segs[0].W, segs[0].y, segs[0].rows, segs[0].dtype = Wd.ptr, y.ptr, rows, dt
            d = _lib.GemmDesc()
            d.segs, d.nseg, d.X, d.n_tokens, d.in_features, d.workspace, d.workspace_bytes = segs, 1, Xd.ptr, T, inf, ws.ptr, nbytes
            _lib.check(L.ntk_gemm_quant_f16(C.byref(d), None), "gemm_quant_f16")
        errs.append(float(np.sqrt(np.mean(((y.numpy(np.float32).reshape(T, rows) - want) / size) ** 2))))
    print("rms error over size, a scale per group / per token:", errs)
    assert errs[0] <= 1.1 * errs[1]


@pytest.mark.parametrize("qname", ["Q4_K", "Q5_K", "Q6_K"])
@pytest.mark.parametrize("T,rows,inf", [(2, (16,), 256), (7, (16, 16, 16), 28672), (16, (4096, 80), 1280), (16, (65536,), 256), (9, (43008, 16), 768), (2, (33024,), 1024), (16, (20480, 48, 6000), 1280),
                                        (5, (16400,), 2304), (16, (9216, 4096), 2816), (3, (6160,), 6144)])
def test_products_through_the_decode_repack(qname, T, rows, inf):
    """the repack through either form: with its planes in LDS (few rows) and in registers (gemm_short.hip: many) -- one unit of 256 columns, three, four, five, nine, eleven, 24 over its waves and
    slices, tiles that end inside a batch, several matrices, the norm's 1 / rms, a residual.  Values and bound as above."""
    gt = getattr(G, "GGML_" + qname)
    L, r = lib(), np.random.Generator(np.random.Philox(key=[T, sum(rows) + inf]))
    from ntransformer_amd import ops
    mats, dt = [], None
    for n in rows:
        raw, W, dt = weights(r, gt, n, inf)
        mats.append((ops.rp_pack(DB.from_numpy(raw), n, inf, dt), W))
    assert L.ntk_gemm_short_takes((C.c_int * len(rows))(*rows), len(rows), T, inf, dt)
    nbytes = L.ntk_gemm_quant_workspace_bytes(inf, sum(rows))
    ws = DB.zeros(nbytes)
    X = r.standard_normal((T, inf)).astype(np.float32)
    X[:, 64:320] *= np.float32(1e4)
    X[T // 2, : inf // 2] = 0.0
    X[0] *= np.float32(1e12)
    X[T - 1] *= np.float32(1e-12)

    def go(normed, eps=0.0, resid=None, partials=None):
        ys = [DB.from_numpy(np.full((T, n), 7.0, np.float32)) for n in rows] if resid is None else [resid]
        segs = (_lib.GemvSeg * len(rows))()
        for s, (w, _), y, n in zip(segs, mats, ys, rows):
            s.W, s.y, s.rows, s.dtype = w.ptr, y.ptr, n, dt
        d = _lib.GemmDesc()
        d.segs, d.nseg, d.n_tokens, d.in_features, d.resid, d.weights_repacked = segs, len(rows), T, inf, None if resid is None else resid.ptr, 1
        d.workspace, d.workspace_bytes = ws.ptr, nbytes
        d.partials = C.pointer(partials) if partials is not None else None
        _lib.check(L.ntk_gemm_short(C.byref(d), normed, eps, 0, None), "gemm_short")
        return [y.numpy(np.float32).reshape(T, n).astype(np.float64) for y, n in zip(ys, rows)]
    Xd = DB.from_numpy(X)
    _lib.check(L.ntk_short_prepare_x(Xd.ptr, T, inf, ws.ptr, None), "short_prepare_x")
    x64 = X.astype(np.float64)
    first = go(0)
    for (_, W), y in zip(mats, first):
        close(y, W, x64)
    assert all(np.array_equal(a, b) for a, b in zip(first, go(0)))
    eps, nw = 1e-5, (1.0 + 0.1 * r.standard_normal(inf)).astype(np.float32)
    hd, nd = DB.from_numpy(X), DB.from_numpy(nw)
    _lib.check(L.ntk_short_norm_prepare_x(hd.ptr, None, nd.ptr, T, inf, ws.ptr, None), "short_norm")
    n64 = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + eps) * nw
    for (_, W), y in zip(mats, go(1, eps)):
        close(y, W, n64)
    if len(rows) > 1 or rows[0] % 256:
        return
    W, res, pt = mats[0][1], r.standard_normal((T, rows[0])).astype(np.float32), _lib.GemmPartials()
    got = go(1, eps, DB.from_numpy(res))[0]
    assert (np.abs(got - (res + n64 @ W.T)) <= REL * (np.sqrt((n64 ** 2) @ (W ** 2).T) + np.abs(res))).all()


@pytest.mark.parametrize("qa,qb", [("Q4_K", "Q6_K"), ("Q5_K", "Q4_K"), ("Q6_K", "Q5_K"), ("Q8_0", "Q4_K")])
@pytest.mark.parametrize("T,ra,rb,inf", [(16, (4096, 1024), (1024,), 4096), (2, (16,), (16,), 256), (7, (80,), (4096, 48), 1280), (11, (6160, 1040), (1040,), 2304), (17, (1024,), (512,), 1024)])
def test_two_formats_over_one_workspace(qa, qb, T, ra, rb, inf):
    """one launch for both (K-quants of up to 16 tokens), or one after the other: results as each one's own, the second's sums behind the first's; the bound as above"""
    L, r = lib(), np.random.Generator(np.random.Philox(key=[T, sum(ra) + inf]))
    L.ntk_gemm_short_two.argtypes = [C.POINTER(_lib.GemmDesc)] * 2 + [C.c_int, C.c_float, C.c_size_t, VP]
    from ntransformer_amd import ops
    nbytes = L.ntk_gemm_quant_workspace_bytes(inf, 4 * (sum(ra) + sum(rb)))       # (two launches' sums side by side)
    ws, eps = DB.zeros(nbytes), 1e-5
    X, nw = r.standard_normal((T, inf)).astype(np.float32), (1.0 + 0.1 * r.standard_normal(inf)).astype(np.float32)
    X[:, 64:200] *= np.float32(1e3)
    xd, nd = DB.from_numpy(X), DB.from_numpy(nw)
    _lib.check(L.ntk_short_norm_prepare_x(xd.ptr, None, nd.ptr, T, inf, ws.ptr, None), "short_norm")
    x64 = X.astype(np.float64)
    n64 = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + eps) * nw
    sides, keep = [], []
    for q, rows in ((qa, ra), (qb, rb)):
        mats, pt = [], _lib.GemmPartials()
        segs = (_lib.GemvSeg * len(rows))()
        for s, n in zip(segs, rows):
            raw, W, dt = weights(r, getattr(G, "GGML_" + q), n, inf)
            w = DB.from_numpy(raw) if q == "Q8_0" else ops.rp_pack(DB.from_numpy(raw), n, inf, dt)
            y = DB.from_numpy(np.full((T, n), 7.0, np.float32))
            s.W, s.y, s.rows, s.dtype = w.ptr, y.ptr, n, dt
            mats.append((W, y, n))
            keep.append(w)
        if not L.ntk_gemm_short_takes((C.c_int * len(rows))(*rows), len(rows), T, inf, dt):
            pytest.skip("not a size of this form")
        d = _lib.GemmDesc()
        d.segs, d.nseg, d.n_tokens, d.in_features, d.weights_repacked = segs, len(rows), T, inf, int(q != "Q8_0")
        d.workspace, d.workspace_bytes, d.partials = ws.ptr, nbytes, C.pointer(pt)
        sides.append((d, pt, mats, segs))
    _lib.check(L.ntk_gemm_short_two(C.byref(sides[0][0]), C.byref(sides[1][0]), 1, eps, 0, None), "gemm_short_two")
    whole = ws.numpy(np.float32)
    for d, pt, mats, _ in sides:
        for k, (W, y, n) in enumerate(mats):
            if pt.nsplit > 1:
                at = (pt.part[k] - ws.ptr) // 4
                got = whole[at:at + pt.nsplit * T * n].reshape(pt.nsplit, T, n).astype(np.float64).sum(0)
            else:
                got = y.numpy(np.float32).reshape(T, n).astype(np.float64)
            close(got, W, n64)


# root mean square of the error over the products' size of the form with its planes in LDS, on these values: (normal ones, two draws; with eight channels a
# hundred times the others', 24 draws: how far off such a sum is depends on which products the channels fall into)
LDS_ERROR = {"Q4_K": (1.477e-7, 1.808e-7), "Q5_K": (1.501e-7, 1.805e-7), "Q6_K": (1.122e-7, 1.163e-7)}


@pytest.mark.parametrize("qname", ["Q4_K", "Q5_K", "Q6_K"])
def test_planes_in_registers_lose_no_precision(qname):
    """the form with its planes in registers against 64 bits, by the mean over half a million products a draw: no further off than the other one"""
    import torch
    from ntransformer_amd import ops
    T, rows, inf = 16, 28672, 4096
    gt = getattr(G, "GGML_" + qname)
    L, r = lib(), np.random.Generator(np.random.Philox(key=[7, gt]))
    dt = G.GGML_TO_DT[gt]
    L.ntk_gemm_short_form.argtypes = [C.POINTER(C.c_int)] + [C.c_int] * 5
    assert L.ntk_gemm_short_form((C.c_int * 1)(rows), 1, T, inf, dt, 1) == 2
    raw, W, _ = weights(r, gt, rows, inf)
    w = ops.rp_pack(DB.from_numpy(raw), rows, inf, dt)
    W = torch.from_numpy(W).cuda()
    nbytes = L.ntk_gemm_quant_workspace_bytes(inf, rows)
    ws, y = DB.zeros(nbytes), DB.zeros(T * rows * 4)
    square = [[], []]
    for towers in [False] * 2 + [True] * 24:
        X = r.standard_normal((T, inf)).astype(np.float32)
        if towers:
            X[:, r.permutation(inf)[:8]] *= np.float32(100)
        Xd = DB.from_numpy(X)
        _lib.check(L.ntk_short_prepare_x(Xd.ptr, T, inf, ws.ptr, None), "short_prepare_x")
        segs = (_lib.GemvSeg * 1)()
        segs[0].W, segs[0].y, segs[0].rows, segs[0].dtype = w.ptr, y.ptr, rows, dt
        d = _lib.GemmDesc()
        d.segs, d.nseg, d.n_tokens, d.in_features, d.weights_repacked, d.workspace, d.workspace_bytes = segs, 1, T, inf, 1, ws.ptr, nbytes
        _lib.check(L.ntk_gemm_short(C.byref(d), 0, 0.0, 0, None), "gemm_short")
        x = torch.from_numpy(X.astype(np.float64)).cuda()
        err = (torch.from_numpy(y.numpy(np.float32).reshape(T, rows).astype(np.float64)).cuda() - x @ W.T) / torch.sqrt((x * x) @ (W * W).T)
        square[towers].append(float((err * err).mean()))
    got = [float(np.sqrt(np.mean(v))) for v in square]
    assert got[0] <= LDS_ERROR[qname][0] and got[1] <= LDS_ERROR[qname][1], got


@pytest.mark.parametrize("qname", ["Q4_K", "Q5_K", "Q6_K"])
@pytest.mark.parametrize("rows,inf,form", [(33024, 1024, 2), (48, 1024, 1)])
def test_values_that_are_none_stay_in_their_token(qname, rows, inf, form):
    """NaN and infinities in some tokens, with the planes in registers and in LDS: those tokens' results are none either, the others' bits do not change"""
    from ntransformer_amd import ops
    T, gt = 9, getattr(G, "GGML_" + qname)
    L, r = lib(), np.random.Generator(np.random.Philox(key=[rows, gt]))
    dt = G.GGML_TO_DT[gt]
    L.ntk_gemm_short_form.argtypes = [C.POINTER(C.c_int)] + [C.c_int] * 5
    assert L.ntk_gemm_short_form((C.c_int * 1)(rows), 1, T, inf, dt, 1) == form
    raw = np.frombuffer(G.synth_tensor(r, gt, rows, inf), np.uint8)
    w = ops.rp_pack(DB.from_numpy(raw), rows, inf, dt)
    nbytes = L.ntk_gemm_quant_workspace_bytes(inf, rows)
    ws, y = DB.zeros(nbytes), DB.zeros(T * rows * 4)

    def go(X):
        Xd = DB.from_numpy(X)
        _lib.check(L.ntk_short_prepare_x(Xd.ptr, T, inf, ws.ptr, None), "short_prepare_x")
        segs = (_lib.GemvSeg * 1)()
        segs[0].W, segs[0].y, segs[0].rows, segs[0].dtype = w.ptr, y.ptr, rows, dt
        d = _lib.GemmDesc()
        d.segs, d.nseg, d.n_tokens, d.in_features, d.weights_repacked, d.workspace, d.workspace_bytes = segs, 1, T, inf, 1, ws.ptr, nbytes
        _lib.check(L.ntk_gemm_short(C.byref(d), 0, 0.0, 0, None), "gemm_short")
        return y.numpy(np.float32).reshape(T, rows)
    X = r.standard_normal((T, inf)).astype(np.float32)
    plain = go(X)
    X[2, 700], X[4, 3], X[4, 4], X[8, inf - 1] = np.nan, np.inf, -np.inf, -np.inf
    got = go(X)
    bad = [2, 4, 8]
    assert not np.isfinite(got[bad]).any()
    good = [t for t in range(T) if t not in bad]
    assert np.array_equal(got[good], plain[good])


@pytest.mark.parametrize("qa,qb", [("Q4_K", "Q6_K"), ("Q4_K", "Q5_K"), ("Q5_K", "Q6_K")])
@pytest.mark.parametrize("turned", [False, True])
@pytest.mark.parametrize("T,ra,rb,inf,at,joins", [(16, (4096, 1024), (1024,), 4096, 0, 1), (2, (4096, 1024), (1040,), 4096, 512, 1), (16, (64,), (32,), 512, 0, 0), (17, (4096, 1024), (1024,), 4096, 64, 0)])
def test_two_formats_in_one_launch(qa, qb, turned, T, ra, rb, inf, at, joins):
    """every pair of formats in both orders: in one launch and, for matrices too small and for 17 tokens, in two -- asked for, so that the launch is not left untested; sums behind others in their area"""
    from ntransformer_amd import ops
    L, r = lib(), np.random.Generator(np.random.Philox(key=[T + at, sum(ra) + inf]))
    L.ntk_gemm_short_two.argtypes = [C.POINTER(_lib.GemmDesc)] * 2 + [C.c_int, C.c_float, C.c_size_t, VP]
    L.ntk_gemm_short_two_joins.argtypes = [C.POINTER(_lib.GemmDesc)] * 2 + [C.c_size_t]
    if turned:
        qa, qb = qb, qa
    nbytes = L.ntk_gemm_quant_workspace_bytes(inf, 4 * (sum(ra) + sum(rb)))
    ws, eps = DB.zeros(nbytes), 1e-5
    X, nw = r.standard_normal((T, inf)).astype(np.float32), (1.0 + 0.1 * r.standard_normal(inf)).astype(np.float32)
    xd, nd = DB.from_numpy(X), DB.from_numpy(nw)
    _lib.check(L.ntk_short_norm_prepare_x(xd.ptr, None, nd.ptr, T, inf, ws.ptr, None), "short_norm")
    x64 = X.astype(np.float64)
    n64 = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + eps) * nw
    sides, keep = [], []
    for q, rows in ((qa, ra), (qb, rb)):
        mats, pt, segs = [], _lib.GemmPartials(), (_lib.GemvSeg * len(rows))()
        for s, n in zip(segs, rows):
            raw, W, dt = weights(r, getattr(G, "GGML_" + q), n, inf)
            w, y = ops.rp_pack(DB.from_numpy(raw), n, inf, dt), DB.from_numpy(np.full((T, n), 7.0, np.float32))
            s.W, s.y, s.rows, s.dtype = w.ptr, y.ptr, n, dt
            mats.append((W, y, n))
            keep.append(w)
        if not L.ntk_gemm_short_takes((C.c_int * len(rows))(*rows), len(rows), T, inf, dt):
            assert T > 16 and q == "Q6_K"
            pytest.skip("32 tokens of the format that scales per 16 columns")
        d = _lib.GemmDesc()
        d.segs, d.nseg, d.n_tokens, d.in_features, d.weights_repacked = segs, len(rows), T, inf, 1
        d.workspace, d.workspace_bytes, d.partials = ws.ptr, nbytes, C.pointer(pt)
        sides.append((d, pt, mats, segs))
    a, b = C.byref(sides[0][0]), C.byref(sides[1][0])
    assert L.ntk_gemm_short_two_joins(a, b, at) == joins
    before = ws.numpy(np.float32)
    _lib.check(L.ntk_gemm_short_two(a, b, 1, eps, at, None), "gemm_short_two")
    whole, first = ws.numpy(np.float32), None
    for d, pt, mats, _ in sides:
        for k, (W, y, n) in enumerate(mats):
            if pt.nsplit > 1:
                place = (pt.part[k] - ws.ptr) // 4
                first = place if first is None else min(first, place)
                got = whole[place:place + pt.nsplit * T * n].reshape(pt.nsplit, T, n).astype(np.float64).sum(0)
            else:
                got = y.numpy(np.float32).reshape(T, n).astype(np.float64)
            close(got, W, n64)
    if first is not None and at:
        assert np.array_equal(whole[first - at:first], before[first - at:first])      # (what lies in front in that area)
