"""Launches of a decoded token that stand for two: against the two, bit for bit where no sum changes its order, else within 4e-6 of the results' size (float32 sums in another order).
Ranks that end inside a lane's eight columns and that take the separate launches, states up to and beyond the line, windows, tables and capped products of odd sizes."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import layers as Lr
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu
VP, I, F = C.c_void_p, C.c_int, C.c_float


def bf16(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def weights(g, shape, dtype):
    w = (g.standard_normal(shape) / np.sqrt(shape[-1])).astype(np.float32)
    return (DB.from_numpy(bf16(w)), 9) if dtype == "bf16" else (DB.from_numpy(w), 0)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("T,H,dn,dr,R,dims,layout,pos0", [(1, 16, 128, 64, 512, 64, 1, 37), (3, 2, 16, 8, 32, 8, 0, 0), (8, 3, 24, 10, 70, 6, 1, 5), (2, 1, 40, 0, 64, 0, 0, 9)])
def test_queries_folded_and_turned_beside_the_cache_rows(dtype, T, H, dn, dr, R, dims, layout, pos0):
    L, g = Lr._bind(), np.random.default_rng(T * R)
    L.ntk_latent_fold_query_rotate.argtypes = [VP, VP, I, VP] + [I] * 6 + [C.POINTER(Lr.Rotary), VP, I, VP, I, VP, F, I, VP]
    qd = dn + dr
    q, kv = g.standard_normal((T, H * qd)).astype(np.float32), g.standard_normal((T, R + dr)).astype(np.float32)
    w, wd = weights(g, (H * dn, R), dtype)
    nw = DB.from_numpy((1 + 0.1 * g.standard_normal(R)).astype(np.float32))
    freq = DB.from_numpy(np.power(10000.0, -np.arange(max(dims // 2, 1)) / max(dims // 2, 1)))
    rot = Lr.Rotary(freq.ptr, 1.25, dims, layout)
    kb, out = DB.from_numpy(kv), []
    for one in (0, 1):
        qb, qf, cache = DB.from_numpy(q), DB.zeros(T * H * (R + dr) * 4), DB.from_numpy(np.full((pos0 + T, R + dr), 3.0, np.float32))
        if one:
            Lr.check(L.ntk_latent_fold_query_rotate(qf.ptr, qb.ptr, H * qd, w.ptr, wd, T, H, dn, dr, R, C.byref(rot), cache.ptr, R + dr, kb.ptr, R + dr, nw.ptr, 1e-5, pos0, None), "rotate")
            assert np.array_equal(qb.numpy(np.float32)[:q.size], q.ravel())            # (only read)
        else:
            Lr.check(L.ntk_latent_prepare(cache.ptr, R + dr, kb.ptr, R + dr, nw.ptr, 1e-5, R, dr, qb.ptr, H * qd, H, qd, C.byref(rot), pos0, T, None), "prepare")
            Lr.check(L.ntk_latent_fold_query(qf.ptr, qb.ptr, H * qd, w.ptr, wd, T, H, dn, dr, R, None), "fold")
        out.append((qf.numpy(np.float32), cache.numpy(np.float32)))
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("T,H,R,dr,dv,pos0,window", [(1, 16, 512, 64, 128, 40, 0), (1, 16, 512, 64, 128, 1500, 0), (1, 4, 512, 64, 128, 1600, 0), (2, 3, 64, 16, 40, 700, 0), (8, 2, 72, 8, 17, 170, 0),
                                                   (1, 2, 70, 6, 16, 300, 0), (1, 5, 8, 0, 3, 0, 0), (3, 2, 256, 32, 64, 900, 100)])
def test_states_joined_where_they_are_unfolded(dtype, T, H, R, dr, dv, pos0, window):
    L, g = Lr._bind(), np.random.default_rng(R + pos0)
    L.ntk_latent_attention_unfold.argtypes = [VP, I, VP, I, VP] + [I] * 3 + [VP, VP, VP] + [I] * 7 + [F, VP, VP]
    row = R + dr
    qf, cache = (DB.from_numpy(g.standard_normal(s).astype(np.float32)) for s in ((T, H * row), (pos0 + T, row)))
    w, wd = weights(g, (H * dv, R), dtype)
    gate = DB.from_numpy(g.standard_normal((T, H * dv)).astype(np.float32))
    L.ntk_latent_attention_scratch.restype = C.c_size_t
    n = int(L.ntk_latent_attention_scratch(T, H, R, pos0 + T))
    for head_gate, gp in ((0, gate.ptr), (1, gate.ptr), (0, None)):
        out = []
        for one in (0, 1):
            scr, lat, o = DB.from_numpy(np.full(n, np.nan, np.float32)), DB.zeros(T * H * R * 4), DB.zeros(T * H * dv * 4)
            if one:
                Lr.check(L.ntk_latent_attention_unfold(o.ptr, H * dv, w.ptr, wd, gp, H * dv, head_gate, dv, lat.ptr, qf.ptr, cache.ptr, row, R, dr, H, pos0, T, window, 0.05, scr.ptr, None), "unfold")
            else:
                Lr.check(L.ntk_latent_attention(lat.ptr, H * R, qf.ptr, H * row, None, 0, None, 0, cache.ptr, row, R, dr, H, 1, 1, 1, pos0, T, 0, window, 0.05, scr.ptr, None), "attention")
                Lr.check(L.ntk_latent_unfold_value_ex(o.ptr, H * dv, lat.ptr, w.ptr, wd, gp, H * dv, head_gate, T, H, dv, R, None), "unfold")
            out.append(o.numpy(np.float32))
        assert np.isfinite(out[1]).all() and np.abs(out[0] - out[1]).max() <= 4e-6 * np.abs(out[0]).max()


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("width", [4, 192, 2048, 5000])
def test_rows_of_the_table(dtype, width):
    L, g = Lr._bind(), np.random.default_rng(width)
    L.ntk_embed_token.argtypes = [VP, VP, I, I, I, I, F, VP]
    L.ntk_embed_dense_scaled.argtypes = [VP, VP, I, VP, I, I, I, F, VP]
    x = g.standard_normal((7, width)).astype(np.float32)
    tab = DB.from_numpy(bf16(x)) if dtype == "bf16" else DB.from_numpy(x)
    wd = 9 if dtype == "bf16" else 0
    want = ((bf16(x).astype(np.uint32) << 16).view(np.float32) if dtype == "bf16" else x) * np.float32(1.7)
    toks = [3, 6, 0, 7, 2]                                     # (one past the table: zeros)
    o, at = DB.from_numpy(np.full((5, width), 9.0, np.float32)), DB.from_numpy(np.array(toks, np.int32))
    Lr.check(L.ntk_embed_dense_scaled(o.ptr, tab.ptr, wd, at.ptr, 5, 7, width, 1.7, None), "embed")
    got = o.numpy(np.float32).reshape(5, width)
    for t, k in enumerate(toks):
        assert np.array_equal(got[t], want[k] if k < 7 else np.zeros(width, np.float32))
        Lr.check(L.ntk_embed_token(o.ptr, tab.ptr, wd, k, 7, width, 1.7, None), "embed_token")
        assert np.array_equal(o.numpy(np.float32)[:width], got[t])
    assert L.ntk_embed_token(o.ptr, tab.ptr, wd, 1, 7, 3, 1.0, None) != 0


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("T,N,K", [(1, 1000, 64), (8, 33, 72), (9, 130, 64), (1, 7, 5)])
def test_capped_products(dtype, T, N, K):
    L, g = Lr._bind(), np.random.default_rng(N)
    L.ntk_dense_capped.argtypes = [C.POINTER(Lr.DenseDesc), F, VP]
    x, (w, wd) = DB.from_numpy(g.standard_normal((T, K)).astype(np.float32)), weights(g, (N, K), dtype)
    out = []
    for one in (0, 1):
        y = DB.zeros(T * N * 4)
        d = Lr.DenseDesc()
        d.Y, d.ldy, d.X, d.ldx, d.W, d.wdtype, d.G, d.row_div, d.T, d.N, d.K = y.ptr, N, x.ptr, K, w.ptr, wd, 1, 1, T, N, K
        if one:
            Lr.check(L.ntk_dense_capped(C.byref(d), 1.5, None), "capped")
        else:
            Lr.check(L.ntk_dense(C.byref(d), None), "dense")
            Lr.check(L.ntk_softcap_rows(y.ptr, N, 1.5, T, N, None), "softcap")
        out.append(y.numpy(np.float32)[:T * N])
    assert np.array_equal(*out) and np.abs(out[0]).max() <= 1.5
    d.act = 1
    assert L.ntk_dense_capped(C.byref(d), 1.5, None) != 0


@pytest.mark.parametrize("T,n,E,top", [(1, 2048, 32, 6), (8, 192, 6, 2), (3, 2052, 33, 4), (2, 70, 5, 5), (1, 5000, 200, 8)])
def test_router_of_a_row_normed_in_its_launch(T, n, E, top):
    L, g = Lr._bind(), np.random.default_rng(n)
    L.ntk_moe_norm_route.argtypes = [VP, VP, VP, VP, I, VP, I, VP, F, F, VP, VP] + [I] * 4 + [C.POINTER(Lr.RouteDesc), VP]
    x = DB.from_numpy((3 * g.standard_normal((T, n))).astype(np.float32))
    nw, wr, ws = (DB.from_numpy((0.2 * g.standard_normal(s)).astype(np.float32)) for s in (n, (E, n), n))
    r = Lr.RouteDesc()
    r.score, r.groups, r.renorm, r.scale = 0, 1, 1, 1.0
    out = []
    for one in (0, 1):
        h, ids, wts, sg = DB.zeros(T * n * 4), DB.zeros(T * top * 4), DB.zeros(T * top * 4), DB.zeros(T * 4)
        if one:
            Lr.check(L.ntk_moe_norm_route(ids.ptr, wts.ptr, sg.ptr, h.ptr, n, x.ptr, n, nw.ptr, 1e-5, 1.0, wr.ptr, ws.ptr, T, n, E, top, C.byref(r), None), "norm_route")
        else:
            Lr.check(L.ntk_rmsnorm_offset(h.ptr, nw.ptr, None, None, n, x.ptr, n, T, n, 1e-5, 1.0, None), "norm")
            Lr.check(L.ntk_moe_route_ex(ids.ptr, wts.ptr, sg.ptr, h.ptr, n, wr.ptr, ws.ptr, T, n, E, top, C.byref(r), None), "route")
        out.append((ids.numpy(np.int32)[:T * top], h.numpy(np.float32)[:T * n], wts.numpy(np.float32)[:T * top], sg.numpy(np.float32)[:T]))
    assert np.array_equal(out[0][0], out[1][0])
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.isfinite(b).all() and np.abs(a - b).max() <= 2e-5 * np.abs(a).max()      # (logits of up to 5000 products behind a norm whose sum has another order)


@pytest.mark.parametrize("T,H,R,dr,pos0,n,E,top", [(1, 16, 512, 64, 1100, 2048, 32, 6), (8, 1, 512, 64, 300, 2052, 33, 4), (3, 16, 512, 304, 20, 4096, 256, 8), (2, 5, 328, 8, 9, 70, 5, 5),
                                                 (1, 16, 512, 64, 40, 5000, 32, 6), (2, 4, 256, 32, 90, 512, 12, 3), (1, 4, 330, 6, 90, 512, 12, 3)])
def test_router_beside_attention(T, H, R, dr, pos0, n, E, top):
    """the last three: rows too long for that launch, attention of four waves, keys off 16 bytes -- the router's own launch"""
    L, g = Lr._bind(), np.random.default_rng(n + R)
    L.ntk_latent_attention_unfold.argtypes = [VP, I, VP, I, VP] + [I] * 3 + [VP, VP, VP] + [I] * 7 + [F, VP, VP]
    L.ntk_latent_attention_unfold_route.argtypes = [VP, I, VP, I, VP] + [I] * 3 + [VP, VP, VP] + [I] * 7 + [F, VP, VP, VP]
    L.ntk_moe_norm_route.argtypes = [VP, VP, VP, VP, I, VP, I, VP, F, F, VP, VP] + [I] * 4 + [C.POINTER(Lr.RouteDesc), VP]
    row, dv = R + dr, 24
    qf, cache = (DB.from_numpy(g.standard_normal(s).astype(np.float32)) for s in ((T, H * row), (pos0 + T, row)))
    w, wd = weights(g, (H * dv, R), "bf16")
    L.ntk_latent_attention_scratch.restype = C.c_size_t
    scr = DB.zeros(int(L.ntk_latent_attention_scratch(T, H, R, pos0 + T)) * 4)
    lat = DB.zeros(T * H * R * 4)
    x = DB.from_numpy((3 * g.standard_normal((T, n))).astype(np.float32))
    nw, wr, ws = (DB.from_numpy((0.2 * g.standard_normal(s)).astype(np.float32)) for s in (n, (E, n), n))
    form = Lr.RouteDesc()
    form.score, form.groups, form.renorm, form.scale = 0, 1, 1, 1.0
    out = []
    for one in (0, 1):
        o, h, ids, wts, sg = DB.zeros(T * H * dv * 4), DB.zeros(T * n * 4), DB.zeros(T * top * 4), DB.zeros(T * top * 4), DB.zeros(T * 4)
        att = (o.ptr, H * dv, w.ptr, wd, None, 0, 0, dv, lat.ptr, qf.ptr, cache.ptr, row, R, dr, H, pos0, T, 0, 0.05, scr.ptr)
        if one:
            r = Lr.NormRoute(ids.ptr, wts.ptr, sg.ptr, h.ptr, n, x.ptr, n, nw.ptr, 1e-5, 1.0, wr.ptr, ws.ptr, T, n, E, top, C.pointer(form))
            Lr.check(L.ntk_latent_attention_unfold_route(*att, C.byref(r), None), "beside")
        else:
            Lr.check(L.ntk_latent_attention_unfold(*att, None), "unfold")
            Lr.check(L.ntk_moe_norm_route(ids.ptr, wts.ptr, sg.ptr, h.ptr, n, x.ptr, n, nw.ptr, 1e-5, 1.0, wr.ptr, ws.ptr, T, n, E, top, C.byref(form), None), "route")
        out.append((o.numpy(np.float32), ids.numpy(np.int32)[:T * top], h.numpy(np.float32)[:T * n], wts.numpy(np.float32)[:T * top], sg.numpy(np.float32)[:T]))
    for a, b in zip(out[0][:2], out[1][:2]):
        assert np.array_equal(a, b)
    for a, b in zip(out[0][2:], out[1][2:]):
        assert np.isfinite(b).all() and np.abs(a - b).max() <= 2e-5 * np.abs(a).max()      # (a norm whose sum is of eight waves' parts instead of sixteen in front of up to 4096 products)
    r.top = E + 1
    assert L.ntk_latent_attention_unfold_route(*att, C.byref(r), None) != 0
