"""Products whose operands go from memory straight into LDS (csrc/gemm_direct.hip.h) and the launches that leave rounded activations for them, against float64 over the
rounded inputs.  Bounds: a sum of K products in 32 bits is off by at most (K + 2) 2^-24 of the sum of their sizes; a bfloat16 result by 2^-8 of itself beside that."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _round(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16 << 16).astype(np.uint32).view(np.float32)


def _case(rng, T, N, K, G=0):
    return rng.standard_normal((T, K)).astype(np.float32), _round(rng.standard_normal((G, N, K) if G else (N, K)).astype(np.float32) / np.sqrt(K))


def _close(got, x, w, out=None, bf=False, slack=1.0, f32=False):
    xd, wd = (x if f32 else _round(x)).astype(np.float64), w.astype(np.float64)
    ref = xd @ wd.T
    bound = (x.shape[1] + 2) * U * (np.abs(xd) @ np.abs(wd).T)
    if out is not None:
        ref, bound = out(ref, bound)
    if bf:
        bound = bound + 2.0 ** -8 * (np.abs(ref) + bound)
    assert np.isfinite(got).all()
    assert (np.abs(got - ref) <= slack * bound + 1e-30).all(), float((np.abs(got - ref) / (bound + 1e-30)).max())


# tiles of 64 x 64 .. 256 x 256 and one row, column or chunk less or more; the last three take the large tiles
@pytest.mark.parametrize("T,N,K", [(9, 16, 64), (9, 1, 64), (63, 65, 128), (64, 64, 192), (65, 130, 64), (129, 257, 320), (255, 512, 448), (257, 63, 1024), (300, 4097, 256),
                                   (1000, 6200, 64), (1025, 6300, 192), (1000, 16300, 128)])
def test_direct_products(T, N, K):
    from ntransformer_amd import layers as Lr
    rng = np.random.default_rng(T + N + K)
    x, w = _case(rng, T, N, K)
    _close(Lr.dense_direct(x, w), x, w)
    if T * N < 2e6:
        y0 = rng.standard_normal((T, N)).astype(np.float32)
        _close(Lr.dense_direct(x, w, y0=y0), x, w, lambda r, b: (r + y0, b + 2 * U * (np.abs(y0) + np.abs(r))))
        _close(Lr.dense_direct(x, w, scratch_floats=16 * T * N), x, w, lambda r, b: (r, 2 * b))       # pieces of K
        _close(Lr.dense_direct(x, w, out16=True, act=1), x, w, lambda r, b: (np.maximum(r, 0) ** 2, 2 * np.abs(r) * b + b * b), bf=True)


@pytest.mark.parametrize("T,N,K", [(212, 1536, 2048), (150, 4096, 4096), (500, 3072, 4096)])
def test_five_pieces_of_k(T, N, K):
    """plans of five pieces (64 x 64, 64 x 128 and 128 x 128 tiles): chunks of 64 that they do not share evenly (32 and 64)"""
    from ntransformer_amd import layers as Lr
    x, w = _case(np.random.default_rng(T), T, N, K)
    _close(Lr.dense_direct(x, w, scratch_floats=16 * T * N), x, w, lambda r, b: (r, 2 * b))


@pytest.mark.parametrize("T,ff,K", [(9, 8, 64), (65, 33, 128), (200, 129, 256), (257, 448, 64), (1030, 3111, 64), (1024, 8200, 64)])
@pytest.mark.parametrize("limit,alpha,up,cubic", [(7.0, 1.702, 1.0, 0.0), (float("inf"), 1.0, 0.0, 0.0), (float("inf"), 1.5957691, 0.0, 0.044715)])
def test_gated_units_inside_the_product(T, ff, K, limit, alpha, up, cubic):
    from ntransformer_amd import layers as Lr
    rng = np.random.default_rng(T + ff)
    x, w = _case(rng, T, 2 * ff, K)

    def unit(r, b):
        g, u = np.minimum(r[:, :ff], limit), np.clip(r[:, ff:], -limit, limit)
        s = 1.0 / (1.0 + np.exp(-alpha * (g + cubic * g ** 3)))
        # both factors off by their product's bound (the gate's slope is below 1.2), and a few roundings of the unit itself
        return g * s * (u + up), 1.2 * b[:, :ff] * (np.abs(u + up) + b[:, ff:]) + np.abs(g) * b[:, ff:] + 16 * U * np.abs(g) * (np.abs(u) + 1.0)
    kw = dict(glu_limit=limit, glu_alpha=alpha, glu_up_offset=up, glu_cubic=cubic)
    _close(Lr.dense_direct(x, w, out16=True, **kw), x, w, unit, bf=True)
    _close(Lr.dense_direct(x, w, **kw), x, w, unit)
    if T < 1000:
        w32 = w + rng.standard_normal(w.shape).astype(np.float32) / 1000
        _close(Lr.dense_direct(x, w32, dtype="float32", **kw), x, w32, unit, f32=True)


@pytest.mark.parametrize("T,N,K,ld", [(9, 1, 32, 32), (31, 65, 64, 68), (33, 64, 96, 96), (150, 200, 2048, 2048), (65, 130, 1000, 1000), (200, 700, 416, 1000)])
def test_float32_products(T, N, K, ld):
    from ntransformer_amd import layers as Lr
    rng = np.random.default_rng(T + N)
    x, w = rng.standard_normal((T, ld)).astype(np.float32), (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32)
    if K % 32 == 0:
        _close(Lr.dense_direct(x, w, dtype="float32"), x[:, :K], w, f32=True)
    y0 = rng.standard_normal((T, N)).astype(np.float32)
    _close(Lr.dense(x, w, "float32", scratch_floats=16 * T * N), x[:, :K], w, lambda r, b: (r, 2 * b), f32=True)
    _close(Lr.dense(x, w, "float32", y0=y0), x[:, :K], w, lambda r, b: (r + y0, b + 2 * U * (np.abs(y0) + np.abs(r))), f32=True)
    off = [0, T // 3, T // 3, T - 2]
    ws = np.stack([w, w + 1, w * 2]).astype(np.float32)
    got = Lr.dense(x, ws, "float32", offsets=off)
    for g in range(3):
        if off[g + 1] > off[g]:
            _close(got[off[g]:off[g + 1]], x[off[g]:off[g + 1], :K], ws[g], f32=True)


@pytest.mark.parametrize("counts", [[0, 1, 64, 65, 0, 130], [300, 0, 0, 3], [255, 256, 257, 1], [17] * 70])
def test_groups_and_gathered_rows(counts):
    from ntransformer_amd import layers as Lr
    rng = np.random.default_rng(len(counts))
    T, N, K, G, div = sum(counts), 200, 128, len(counts), 3
    x, w = _case(rng, (T + div - 1) // div, N, K, G)
    rows, off = rng.permutation(T), np.concatenate([[0], np.cumsum(counts)])
    got = Lr.dense_direct(x, w, offsets=off, rows=rows, row_div=div)
    same = Lr.dense_direct(x[rows // div], w, offsets=off)
    extra = Lr.dense_direct(x[rows // div], w, offsets=np.minimum(off, T - 5), fill=3.0)                   # rows that belong to no group stay as they are
    assert np.array_equal(got, same) and (extra[T - 5:] == 3.0).all() and np.array_equal(extra[:T - 5], got[:T - 5])
    for g in range(G):
        if counts[g]:
            _close(got[off[g]:off[g + 1]], x[rows[off[g]:off[g + 1]] // div], w[g])


@pytest.mark.parametrize("T,N,K,ld", [(40, 2048, 1024, 1028), (200, 1500, 512, 512), (1000, 2048, 2048, 2112), (300, 700, 1000, 1000)])
def test_the_product_with_room_for_rounded_activations_equals_the_one_without(T, N, K, ld):
    """one chain of matrix instructions over the inputs in both: the same bits, unless the inputs are cut into pieces"""
    from ntransformer_amd import layers as Lr
    rng = np.random.default_rng(N)
    x = rng.standard_normal((T, ld)).astype(np.float32)
    w = _round(rng.standard_normal((N, K)).astype(np.float32) / np.sqrt(K))
    x[3, 5], x[5, 7] = np.inf, np.nan
    a = Lr.dense(x, w, "bfloat16")
    b = Lr.dense(x, w, "bfloat16", scratch_floats=T * K // 2 + 4)              # room for the rounded rows alone
    assert np.array_equal(np.isfinite(a), np.isfinite(b)) and not np.isfinite(b[[3, 5]]).any()
    assert np.array_equal(np.nan_to_num(a), np.nan_to_num(b))
    c = Lr.dense(x, w, "bfloat16", scratch_floats=T * K // 2 + 8 * T * N)
    fin = np.delete(np.arange(T), [3, 5])
    _close(c[fin], x[fin, :K], w, lambda r, e: (r, 2 * e))


def test_rounding_and_what_is_refused():
    from ntransformer_amd import layers as Lr
    rng = np.random.default_rng(0)
    for T, ld, n in ((3, 16, 16), (70, 100, 96), (9, 37, 37), (5, 40, 33)):
        x = rng.standard_normal((T, ld)).astype(np.float32)
        assert np.array_equal(Lr.round_rows(x, n), _round(x[:, :n]))
    for T, K in ((8, 64), (20, 96)):           # few rows; no whole chunks of inputs
        with pytest.raises(Exception):
            Lr.dense_direct(rng.standard_normal((T, K)).astype(np.float32), np.ones((16, K), np.float32))


@pytest.mark.parametrize("T,n", [(1, 4), (9, 64), (33, 1020), (40, 2048), (9, 4096)])
def test_norms_that_leave_rounded_rows(T, n):
    from ntransformer_amd import layers as Lr
    rng = np.random.default_rng(n)
    x, y = rng.standard_normal((2, T, n)).astype(np.float32)
    w, aw = rng.standard_normal((2, n)).astype(np.float32)
    # (another order of the row's sum: a rounded value may fall to the other side)
    near = lambda got, want: (np.abs(got - want) <= 2.0 ** -7 * np.abs(want) + 1e-30).all()
    a, b, c = Lr.rmsnorm_offset_16(x, w, aw, 1e-5, 1.0)
    p, q = Lr.rmsnorm_offset(x, w, aw, 1e-5, 1.0)
    assert near(a, p) and np.allclose(b, q, rtol=2e-6, atol=0) and np.array_equal(c, _round(b))
    for add in (None, y):
        gx, gh = Lr.rms_seam_16(x, w, 1e-5, add, aw if add is not None else None, 0.7)
        sx, sh = Lr.rms_seam(x, w, 1e-5, add, aw if add is not None else None, 0.7)
        assert np.allclose(gx, sx, rtol=2e-6, atol=2e-6) and near(gh, sh)
    with pytest.raises(Exception):
        Lr.rms_seam_16(rng.standard_normal((2, 4100)).astype(np.float32), np.ones(4100, np.float32), 1e-5)


# bfloat16 keeps eight bits: half a step is 2^-8 of a value; the float32 before it (a mean of up to 256 squares, an exponential) is a few steps of 2^-24 off
def _rounded_near(got, want):
    return (np.abs(got - want) <= (2.0 ** -8 + 64 * 2.0 ** -24) * np.abs(want) + 1e-30).all()


@pytest.mark.parametrize("T,heads,dim,act,shared", [(1, 1, 4, 2, True), (33, 3, 60, 1, False), (40, 5, 64, 2, True), (9, 7, 68, 0, True), (70, 16, 128, 2, True), (5, 3, 132, 1, False), (33, 2, 256, 2, False)])
def test_head_norms_that_leave_rounded_rows(T, heads, dim, act, shared):
    from ntransformer_amd import layers as Lr
    rng = np.random.default_rng(dim)
    n = heads * dim
    x, g = rng.standard_normal((2, T, n + 8)).astype(np.float32)
    w = rng.standard_normal(dim if shared else (heads, dim)).astype(np.float32)
    v = x[:, :n].astype(np.float64).reshape(T, heads, dim)
    c = g[:, :n].astype(np.float64).reshape(T, heads, dim)
    s = 1 / (1 + np.exp(-c))
    want = v / np.sqrt((v * v).mean(-1, keepdims=True) + 1e-5) * w * (s * c if act == 2 else s if act else 1.0) * 0.7
    assert _rounded_near(Lr.head_rmsnorm_gate_16(x, w, g if act else None, act, 0.7, heads, dim, 1e-5), want.reshape(T, n))
    with pytest.raises(Exception):                   # no fours; a head of more than a wave
        Lr.head_rmsnorm_gate_16(x[:, :6].copy(), w.reshape(-1)[:2].copy(), None, 0, 1.0, 1, 2, 1e-5)
    with pytest.raises(Exception):
        Lr.head_rmsnorm_gate_16(rng.standard_normal((2, 260)).astype(np.float32), np.ones(260, np.float32), None, 0, 1.0, 1, 260, 1e-5)


@pytest.mark.parametrize("T,n,per_head", [(1, 4, 0), (33, 1020, 0), (9, 1028, 0), (40, 2048, 128), (5, 24, 4), (70, 2112, 192)])
def test_gates_that_leave_rounded_rows(T, n, per_head):
    from ntransformer_amd import layers as Lr
    rng = np.random.default_rng(n)
    x = rng.standard_normal((T, n + 4)).astype(np.float32)
    g = rng.standard_normal((T, n // per_head + 3 if per_head else n + 8)).astype(np.float32) * 4
    s = 1 / (1 + np.exp(-g.astype(np.float64)))
    s = np.repeat(s[:, :n // per_head], per_head, axis=1) if per_head else s[:, :n]
    assert _rounded_near(Lr.gate_rows_16(x, g, n, per_head), x[:, :n] * s)
    with pytest.raises(Exception):
        Lr.gate_rows_16(x, g, 3, 0)


@pytest.mark.parametrize("T,N,K,tile", [(20, 3264, 2112, (64, 64, 3)), (14, 12320, 4096, (64, 128, 2)), (65, 5504, 6464, (128, 128, 1)), (65, 10976, 6464, (128, 256, 1)),
                                        (200, 5408, 6464, (256, 128, 1)), (129, 10976, 6464, (256, 256, 1))])
def test_five_pieces_of_k_by_their_plans(T, N, K, tile):
    """every tile that takes five pieces, chunks of 64 that they do not share evenly (33, 64 and 101): the plan is asked for, so that another choice does not leave the form untested"""
    from ntransformer_amd import layers as Lr
    import ctypes as C
    plan, f = (C.c_int * 4)(), Lr._bind().ntk_dense_direct_plan
    f.argtypes, f.restype = [C.c_int] * 4 + [C.c_longlong, C.POINTER(C.c_int)], C.c_int
    assert f(T, 1, N, K, 16 * T * N, plan) == 0 and tuple(plan) == tile + (5,)
    x, w = _case(np.random.default_rng(T), T, N, K)
    _close(Lr.dense_direct(x, w, scratch_floats=16 * T * N), x, w)
