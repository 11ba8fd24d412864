"""The tiled products (csrc/gemm_tile.hip.h) at the sizes where a tile, a chunk of inputs or a piece of a split can go wrong, against float64 sums of the values the
matrix cores multiply.  Bound: every one of the K products and additions rounds to 32 bits once, |error| <= (K + 16) * 2^-24 * sum |x w|."""
import numpy as np
import pytest

from ntransformer_amd import layers as Lr

pytestmark = pytest.mark.gpu


def bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32).view(np.float32)


def within_bound(y, x, w, y0=0.0):
    x, w = x.astype(np.float64), w.astype(np.float64)
    bound = (x.shape[1] + 16) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T + np.abs(y0)) + 1e-30
    return np.all(np.abs(y - (y0 + x @ w.T)) <= bound)


def values(dtype, T, N, K, seed):
    g = np.random.default_rng(seed)
    x, w = g.standard_normal((T, K)).astype(np.float32), bf16(g.standard_normal((N, K)) / np.sqrt(K))
    return x, w, (bf16(x) if dtype == "bfloat16" else x)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("T,N,K", [(9, 1, 8), (9, 64, 64), (31, 63, 72), (32, 65, 128), (33, 130, 520), (64, 64, 2048), (65, 516, 2056), (128, 128, 32), (129, 257, 96), (200, 640, 1000),
                                   (300, 2048, 64), (1025, 1028, 40), (12, 3, 4104), (40, 2048, 1536), (17, 100, 37), (70, 33, 515),
                                   (9, 64, 4), (33, 65, 36), (129, 130, 1004), (40, 516, 2044)])     # (rows of four but not of eight: pieces of four weights, float32 only)
def test_edges_of_tiles_chunks_and_pieces(dtype, T, N, K):
    x, w, xr = values(dtype, T, N, K, T * 7 + N)
    for room in (0, 2 * T * N, 16 * T * N):
        assert within_bound(Lr.dense(x, w, dtype, scratch_floats=room), xr, w), room
        y0 = np.random.default_rng(3).standard_normal((T, N)).astype(np.float32)
        assert within_bound(Lr.dense(x, w, dtype, y0=y0, scratch_floats=room), xr, w, y0), room


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("sizes", [(0, 9, 0, 1), (130, 0, 64, 63, 1), (1,) * 70, (0, 0, 300), (5, 200, 31, 33, 0, 129)])
def test_groups_of_every_size(dtype, sizes):
    G, K, N = len(sizes), 104, 96
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    T = int(off[-1])
    x, _, xr = values(dtype, T, 1, K, 5)
    w = bf16(np.random.default_rng(6).standard_normal((G, N, K)))
    order = np.random.default_rng(7).permutation(T).astype(np.int32)
    y = Lr.dense(x, w, dtype, offsets=off, rows=order, row_div=1)
    for g in range(G):
        s = slice(off[g], off[g + 1])
        assert within_bound(y[s], xr[order[s]], w[g]), g


@pytest.mark.parametrize("T,N,K", [(9, 1, 8), (33, 65, 72), (48, 130, 520), (64, 64, 2056), (17, 100, 37), (12, 3, 4104), (70, 33, 515)])
def test_activations_in_three_pieces(T, N, K):
    """bfloat16 weights beside 32-bit activations at the edges of the tile, alone and in groups; rows of every magnitude; what is not finite stays in its row"""
    x, w, _ = values("bfloat16", T, N, K, T + K)
    x *= np.logspace(-25, 25, T).astype(np.float32)[:, None]
    x[:, ::16] *= 3000.0
    assert within_bound(Lr.dense(x, w, "bfloat16", full_x=True), x, w)
    off = np.array([0, T // 3, T // 3, T], np.int32)
    ws, order = bf16(np.random.default_rng(8).standard_normal((3, N, K))), np.random.default_rng(9).permutation(T).astype(np.int32)
    y = Lr.dense(x, ws, "bfloat16", offsets=off, rows=order, row_div=1, full_x=True)
    for g in range(3):
        s = slice(off[g], off[g + 1])
        assert within_bound(y[s], x[order[s]], ws[g]), g
    x[3, 5], x[6, 2], x[7, 0] = np.inf, np.nan, 3.4028235e38
    x[7, 1:] = 0.0
    y = Lr.dense(x, w, "bfloat16", full_x=True)
    keep = [r for r in range(T) if r not in (3, 6)]
    assert within_bound(y[keep], x[keep], w) and np.isnan(y[6]).all() and not np.isfinite(y[3]).any()


@pytest.mark.parametrize("K", [1408, 2048, 4096])
def test_three_pieces_no_further_from_float64_than_a_few_rows(K):
    """root mean square over 24576 results; the products of up to eight rows multiply in 32 bits on the vector units"""
    x, w, _ = values("bfloat16", 48, 512, K, K)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    few = np.concatenate([Lr.dense(x[i:i + 8], w, "bfloat16") for i in range(0, 48, 8)])
    assert np.linalg.norm(Lr.dense(x, w, "bfloat16", full_x=True) - want) <= np.linalg.norm(few - want)


@pytest.mark.parametrize("T,N,K", [(833, 3841, 33), (1025, 3329, 40), (1600, 2049, 67)])
def test_odd_sizes_in_many_tiles(T, N, K):
    """element by element into the larger tiles (K = 40: rows that do not start on 16 bytes), alone and over rows in groups"""
    x, w, xr = values("bfloat16", T, N, K, T)
    if K == 40:
        x = np.concatenate([x, np.full((T, 1), np.nan, np.float32)], axis=1)
    assert within_bound(Lr.dense(x, w, "bfloat16"), xr, w)
    sizes = (T // 2 + 3, 0, 129, T - T // 2 - 132)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    ws = bf16(np.random.default_rng(8).standard_normal((4, N, K)))
    y = Lr.dense(x, ws, "bfloat16", offsets=off)
    for g in range(4):
        s = slice(off[g], off[g + 1])
        assert within_bound(y[s], xr[s], ws[g]), g


def test_an_activation_on_sums_of_pieces():
    x, w, xr = values("bfloat16", 40, 256, 4096, 1)
    y = Lr.dense(x, w, "bfloat16", act=Lr.ACT_RELU2, scratch_floats=16 * 40 * 256)
    z = np.maximum(Lr.dense(x, w, "bfloat16", scratch_floats=16 * 40 * 256), 0.0)
    assert np.array_equal(y, z * z)
