"""ntk_gemm_half (prompt projections over half-precision weights) at the edges of its tiles, chunks and pieces, against float64 sums.  Bound: an activation is off by 2^-23 of its
value at most (what its row's largest adds, 2^-39, is below that here), the K additions round to 32 bits once each, those of runs and pieces once more:
|error| <= (K + 18) * 2^-24 * sum |x w|."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib, ops
from ntransformer_amd import gguf as G

pytestmark = pytest.mark.gpu


def bound():
    """the library with these entry points' types (an unbound call would cut its pointers to 32 bits)"""
    L = _lib.lib()
    L.ntk_gemm_half_workspace_bytes.restype = C.c_size_t
    L.ntk_gemm_half.argtypes = [C.c_void_p] * 3 + [C.c_int] * 4 + [C.c_void_p, C.c_void_p, C.c_size_t, C.c_void_p]
    return L


def run(x, w, y0=None, room=0, given_max=False):
    L = bound()
    T, K = x.shape
    N = w.shape[0]
    need = int(L.ntk_gemm_half_workspace_bytes(T))
    xb, wb = ops.DeviceBuffer.from_numpy(x.astype(np.float32)), ops.DeviceBuffer.from_numpy(w.astype(np.float16))
    yb = ops.DeviceBuffer.from_numpy(y0 if y0 is not None else np.full((T, N), 7.0, np.float32))
    ws = ops.DeviceBuffer(need + room * 4)
    mb = ops.DeviceBuffer.from_numpy(np.abs(x).max(1).astype(np.float32)) if given_max else None
    _lib.check(L.ntk_gemm_half(yb.ptr, wb.ptr, xb.ptr, T, N, K, int(y0 is not None), mb.ptr if mb else None, ws.ptr, need + room * 4, None), "ntk_gemm_half")
    return yb.numpy(np.float32, T * N).reshape(T, N)


def within_bound(y, x, w, y0=0.0):
    x, w = x.astype(np.float64), w.astype(np.float64)
    return np.all(np.abs(y - (y0 + x @ w.T)) <= (x.shape[1] + 18) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T + np.abs(y0)) + 1e-37)


def values(T, N, K, seed):
    g = np.random.default_rng(seed)
    return g.standard_normal((T, K)).astype(np.float32), (g.standard_normal((N, K)) / np.sqrt(K)).astype(np.float16).astype(np.float32)


@pytest.mark.parametrize("T,N,K", [(2, 64, 64), (3, 1, 8), (16, 1024, 4096), (31, 65, 72), (33, 516, 520), (65, 128, 2048), (129, 300, 40), (200, 2048, 1024), (257, 512, 96), (5, 70, 37),
                                   (2, 28672, 128), (1030, 260, 264)])
def test_edges_of_tiles_chunks_and_pieces(T, N, K):
    x, w = values(T, N, K, T + N)
    for room in (0, 16 * T * N):
        assert within_bound(run(x, w, room=room), x, w)
        y0 = np.random.default_rng(2).standard_normal((T, N)).astype(np.float32)
        assert within_bound(run(x, w, y0=y0, room=room, given_max=True), x, w, y0)


def test_rows_of_every_magnitude():
    x, w = values(40, 96, 256, 9)
    x *= np.logspace(-30, 30, 40).astype(np.float32)[:, None]
    x[:, ::16] *= 4000.0                       # a few channels tower over the others
    x[7] = 0.0
    assert within_bound(run(x, w), x, w)


@pytest.mark.parametrize("K", [3072, 3584, 4096, 14336])
@pytest.mark.parametrize("towering", [False, True])
def test_no_further_from_float64_than_the_one_token_products(K, towering):
    """root mean square over 20480 results each, so known to 0.5 %; the lengths from which a prompt takes the tiles (at 3072 with towering channels both are 1.42e-7 .. 1.43e-7: hence 1.03)"""
    x, w = values(40, 512, K, K)
    if towering:
        x[:, ::37] *= 300.0
    want = x.astype(np.float64) @ w.astype(np.float64).T
    xb, wb, yb = ops.DeviceBuffer.from_numpy(x), ops.DeviceBuffer.from_numpy(w.astype(np.float16)), ops.DeviceBuffer(40 * 512 * 4)
    for t in range(40):
        ops.launch_gemv(yb.at(t * 512 * 4), wb, xb.at(t * K * 4), 512, K, G.DT_F16)
    y1 = yb.numpy(np.float32, 40 * 512).reshape(40, 512)
    for room in (0, 16 * 40 * 512):
        assert np.linalg.norm(run(x, w, room=room) - want) <= 1.03 * np.linalg.norm(y1 - want), room


def test_infinities_stay_in_their_row():
    x, w = values(9, 64, 128, 4)
    x[3, 5], x[6, 9] = np.inf, np.nan
    y = run(x, w)
    rows = [r for r in range(9) if r not in (3, 6)]
    assert within_bound(y[rows], x[rows], w) and np.isnan(y[6]).all()
    assert np.array_equal(y[3], np.where(w[:, 5] == 0, np.nan, np.sign(w[:, 5]) * np.inf).astype(np.float32), equal_nan=True)


def test_large_values_beside_an_infinity_and_rows_of_subnormals():
    """a row with an infinity: its finite values stay finite, whatever their size, so every result has the infinity's sign; a row whose largest value is subnormal is not lost"""
    x, w = values(9, 64, 128, 6)
    x[3, 5] = np.inf
    x[3, 20:28] = np.array([7e4, -7e4, 1e9, -1e9, 3e38, -3e38, 65520.0, -65520.0], np.float32)
    x[5] *= np.float32(2.0 ** -128)
    for given_max in (False, True):
        y = run(x, w, given_max=given_max)
        assert np.array_equal(y[3], np.where(w[:, 5] == 0, np.nan, np.sign(w[:, 5]) * np.inf).astype(np.float32), equal_nan=True)
        want = x[5].astype(np.float64) @ w.T.astype(np.float64)
        assert np.abs(y[5] - want).max() < 1e-3 * np.abs(want).max()
        rows = [r for r in range(9) if r not in (3, 5)]
        assert within_bound(y[rows], x[rows], w)


def test_what_it_refuses():
    L = _lib.lib()
    b = ops.DeviceBuffer(4096)
    f = L.ntk_gemm_half
    f.argtypes = [C.c_void_p] * 3 + [C.c_int] * 4 + [C.c_void_p, C.c_void_p, C.c_size_t, C.c_void_p]
    assert f(b.ptr, b.ptr, None, 2, 8, 8, 0, None, b.ptr, 4096, None) == -5
    assert f(b.ptr, b.ptr, b.ptr, 2, 8, 8, 0, None, None, 0, None) == -5 and f(b.ptr, b.ptr, b.ptr, 9, 8, 8, 0, None, b.ptr, 32, None) == -2
    assert f(b.ptr, b.ptr, b.ptr, 2, 0, 8, 0, None, b.ptr, 4096, None) == -2 and f(b.ptr, b.ptr, b.ptr, 0, 8, 8, 0, None, b.ptr, 4096, None) == 0


def test_a_workspace_for_a_few_rows_is_no_slower_than_the_smallest():
    """activations go in pieces of what the workspace holds only where that pays: 200 tokens through a workspace for 16 took seven times as long as through none"""
    import time
    L = bound()
    T, N, K = 200, 4096, 4096
    x, w = ops.DeviceBuffer.zeros(T * K * 4), ops.DeviceBuffer.zeros(N * K * 2)
    y = ops.DeviceBuffer(T * N * 4)
    best = {}
    for rows in (0, 16, 50):
        size = int(L.ntk_gemm_half_workspace_bytes(T)) + rows * (4 * K + 4)
        ws = ops.DeviceBuffer(size)
        for _ in range(6):
            t0 = time.perf_counter()
            for _ in range(30):
                _lib.check(L.ntk_gemm_half(y.ptr, w.ptr, x.ptr, T, N, K, 0, None, ws.ptr, size, None), "ntk_gemm_half")
            _lib.check(L.ntk_stream_synchronize(None), "synchronize")
            best[rows] = min(best.get(rows, 1e9), time.perf_counter() - t0)
    print({r: "%.0f us" % (t / 30 * 1e6) for r, t in best.items()})
    assert max(best[16], best[50]) < 2.0 * best[0]
