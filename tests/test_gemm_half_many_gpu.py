"""ntk_gemm_half_many (several half-precision matrices over one prompt's activations, their gated unit inside the launch) at the edges of its tiles and passes, against float64.
Bound of a product: |error| <= (K + 18) * 2^-24 * sum |x w| (an activation is off by 2^-23 of its value, the K additions round once each, those of runs and pieces once more)."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib, ops

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


class Desc(C.Structure):
    _fields_ = [("W", C.c_void_p * 3), ("Y", C.c_void_p * 3), ("out", C.c_int * 3), ("n", C.c_int), ("X", C.c_void_p), ("n_tokens", C.c_int), ("in_features", C.c_int), ("accumulate", C.c_int),
                ("row_max", C.c_void_p), ("silu", C.c_int), ("workspace", C.c_void_p), ("workspace_bytes", C.c_size_t)]


def run(x, ws, silu=False, room=0, rows_of_a_pass=None, given_max=False):
    L = _lib.lib()
    L.ntk_gemm_half_many.argtypes = [C.POINTER(Desc), C.c_void_p]
    T, K = x.shape
    xb = ops.DeviceBuffer.from_numpy(x)
    # the matrices in one allocation, the second one first (any order is allowed)
    order = [1, 0, 2][:len(ws)] if len(ws) > 1 else [0]
    at, parts, flat = {}, 0, []
    for i in order:
        at[i] = parts
        flat.append(ws[i].astype(np.float16).reshape(-1))
        flat.append(np.zeros((-flat[-1].size) % 8, np.float16))
        parts += flat[-1].size + flat[-2].size
    wb = ops.DeviceBuffer.from_numpy(np.concatenate(flat))
    ys = [ops.DeviceBuffer.from_numpy(np.full((T, w.shape[0]), 7.0, np.float32)) for w in ws]
    d = Desc()
    for i, w in enumerate(ws):
        d.W[i], d.Y[i], d.out[i] = wb.at(2 * at[i]), ys[i].ptr, w.shape[0]
    d.n, d.X, d.n_tokens, d.in_features, d.silu = len(ws), xb.ptr, T, K, int(silu)
    mb = ops.DeviceBuffer.from_numpy(np.abs(x).max(1)) if given_max else None
    d.row_max = mb.ptr if mb else None
    size = (rows_of_a_pass or T) * (K * 4 + 4) + 32 + room * 4
    space = ops.DeviceBuffer(size)
    d.workspace, d.workspace_bytes = space.ptr, size
    _lib.check(L.ntk_gemm_half_many(C.byref(d), None), "ntk_gemm_half_many")
    out = [y.numpy(np.float32, T * w.shape[0]).reshape(T, -1) for y, w in zip(ys, ws)]
    return out[0] if silu else out


def values(T, K, outs, seed):
    g = np.random.default_rng(seed)
    return g.standard_normal((T, K)).astype(np.float32), [(g.standard_normal((n, K)) / np.sqrt(K)).astype(np.float16).astype(np.float32) for n in outs]


def product(x, w):
    x, w = x.astype(np.float64), w.astype(np.float64)
    return x @ w.T, (x.shape[1] + 18) * U * (np.abs(x) @ np.abs(w).T) + 1e-37


@pytest.mark.parametrize("T,K,outs", [(2, 64, (64, 16, 16)), (16, 1024, (300, 65, 1)), (65, 128, (1, 130)), (129, 320, (257, 64, 63)), (200, 4096, (512, 128, 128)), (40, 192, (4100, 3, 260)),
                                      (130, 64, (16500, 260, 250))])
def test_matrices_side_by_side(T, K, outs):
    x, ws = values(T, K, outs, T + K)
    for kw in (dict(), dict(room=16 * T * sum(outs), given_max=True), dict(rows_of_a_pass=max(16, T // 3))):
        for y, w in zip(run(x, ws, **kw), ws):
            want, bound = product(x, w)
            assert (np.abs(y - want) <= bound).all(), kw


@pytest.mark.parametrize("T,K,ff", [(2, 64, 16), (33, 128, 130), (70, 512, 65), (200, 4096, 384), (100, 64, 16400)])
def test_gated_unit_in_the_launch(T, K, ff):
    x, ws = values(T, K, (ff, ff), T + ff)
    for kw in (dict(), dict(given_max=True, rows_of_a_pass=max(16, T // 2))):
        y = run(x, ws, silu=True, **kw)
        (g, bg), (u, bu) = product(x, ws[0]), product(x, ws[1])
        s = 1.0 / (1.0 + np.exp(-g))
        # the unit's slope in the gate is below 1.1; a few roundings of its own
        bound = 1.1 * bg * (np.abs(u) + bu) + np.abs(g * s) * bu + 16 * U * np.abs(g * s * u) + 1e-37
        assert (np.abs(y - g * s * u) <= bound).all()


@pytest.mark.parametrize("T", [129, 144, 145, 161, 200, 257, 300])
def test_rows_shared_evenly_over_tiles(T):
    """the 128 x 256 form (28672 columns: it is the estimate's choice) where its row tiles are not full: 5 and 4 sixteens of 128 rows, odd counts, a last row of its own, three tiles"""
    x, ws = values(T, 1024, (14336, 14336), T)
    y = run(x, ws, silu=True)
    (g, bg), (u, bu) = product(x, ws[0]), product(x, ws[1])
    s = 1.0 / (1.0 + np.exp(-g))
    assert (np.abs(y - g * s * u) <= 1.1 * bg * (np.abs(u) + bu) + np.abs(g * s) * bu + 16 * U * np.abs(g * s * u) + 1e-37).all()


@pytest.mark.parametrize("T,K,outs", [(256, 4096, (4096, 1024, 1024)), (150, 2048, (2048,)), (70, 4160, (6100, 33, 10))])
def test_five_pieces_of_k(T, K, outs):
    """128 x 256, 64 x 64 and 64 x 128 tiles in five pieces, the last of them shorter (64, 32 and 65 chunks)"""
    x, ws = values(T, K, outs, T + K)
    for y, w in zip(run(x, ws, room=16 * T * sum(outs)), ws):
        want, bound = product(x, w)
        assert (np.abs(y - want) <= bound).all()


def test_a_row_that_is_not_finite_and_what_is_refused():
    x, ws = values(20, 128, (70, 70), 3)
    x[4, 9], x[6, 1] = np.nan, np.inf
    y = run(x, ws, silu=True)
    rows = [r for r in range(20) if r not in (4, 6)]
    assert np.array_equal(y[rows], run(x[rows], ws, silu=True)) and np.isnan(y[4]).all()
    L = _lib.lib()
    L.ntk_gemm_half_many.argtypes = [C.POINTER(Desc), C.c_void_p]
    b = ops.DeviceBuffer(1 << 16)
    d = Desc()
    d.W[0] = d.W[1] = d.Y[0] = d.Y[1] = d.X = d.workspace = b.ptr
    d.out[0] = d.out[1] = 8
    d.n, d.n_tokens, d.in_features, d.workspace_bytes = 1, 2, 64, 1 << 16
    call = lambda: L.ntk_gemm_half_many(C.byref(d), None)
    for name, bad, code in (("in_features", 72, -2), ("workspace_bytes", 100, -2), ("n", 4, -5), ("X", None, -5), ("workspace", None, -5)):
        keep = getattr(d, name)
        setattr(d, name, bad)
        assert call() == code, name
        setattr(d, name, keep)
    d.n, d.accumulate = 2, 1
    assert call() == -2
    d.accumulate, d.silu, d.out[1] = 0, 1, 16
    assert call() == -2


def plan(rows, N, K, room):
    out, f = (C.c_int * 4)(), _lib.lib().ntk_gemm_half_plan
    f.argtypes, f.restype = [C.c_int] * 3 + [C.c_longlong, C.POINTER(C.c_int)], C.c_int
    assert f(rows, N, K, room, out) == 0
    return tuple(out)


@pytest.mark.parametrize("T,K,outs,tile", [(14, 2112, (5504,), (64, 64, 2)), (70, 2112, (6100, 33, 11), (64, 128, 2)), (200, 4096, (4096, 1024, 1024), (128, 256, 1))])
def test_five_pieces_of_k_by_their_plans(T, K, outs, tile):
    """every tile in five pieces, the last of them shorter (33 and 64 chunks): the plan is asked for, so that another choice does not leave the form untested"""
    assert plan(T, sum(outs), K, 16 * T * sum(outs)) == tile + (5,)
    x, ws = values(T, K, outs, T + K)
    for y, w in zip(run(x, ws, room=16 * T * sum(outs)), ws):
        want, bound = product(x, w)
        assert (np.abs(y - want) <= bound).all()


@pytest.mark.parametrize("T,ff,K", [(129, 11008, 512), (153, 14336, 512), (257, 7488, 1024), (297, 7488, 1024), (385, 7488, 512)])
def test_rows_shared_evenly_by_their_plans(T, ff, K):
    """two, three and four row tiles of the 128 x 256 form, not all full"""
    assert plan(T, 2 * ff, K, 0) == (128, 256, 1, 1)
    x, ws = values(T, K, (ff, ff), T)
    y = run(x, ws, silu=True)
    (g, bg), (u, bu) = product(x, ws[0]), product(x, ws[1])
    s = 1.0 / (1.0 + np.exp(-g))
    assert (np.abs(y - g * s * u) <= 1.1 * bg * (np.abs(u) + bu) + np.abs(g * s) * bu + 16 * U * np.abs(g * s * u) + 1e-37).all()
