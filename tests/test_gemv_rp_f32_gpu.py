"""ntk_gemv_rp_f32 (one row of F32 activations through a repacked K-quant matrix, F32 products) against float64 over the dequantised weights.  Bound: K additions round once each, the parts of a
16-column run (products, -32 or minimum times the run's sum, scales) a few times more, over the sizes that are added: (in / 64 + 40) * 2^-24 * sum(|q| scale |x|), |q| up to 63."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib
from ntransformer_amd import gguf as G
from ntransformer_amd import ops
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu
KQ = {"Q4_K": G.GGML_Q4_K, "Q5_K": G.GGML_Q5_K, "Q6_K": G.GGML_Q6_K}


def case(gt, rows, n, seed, towering=False):
    g = np.random.Generator(np.random.Philox(key=[20261203, seed]))
    raw = np.frombuffer(G.synth_tensor(g, gt, rows, n), np.uint8)
    x = g.standard_normal(n).astype(np.float32)
    if towering:
        x[::97] *= 300.0
    return raw, G.dequantize(raw, gt, rows * n).reshape(rows, n).astype(np.float64), x


def run(raw, gt, x, rows):
    dt, n = G.GGML_TO_DT[gt], x.size
    rp, xb, yb = ops.rp_pack(DB.from_numpy(raw), rows, n, dt), DB.from_numpy(x), DB.from_numpy(np.full(rows + 3, 7.0, np.float32))
    L = _lib.lib()
    L.ntk_gemv_rp_f32.argtypes = [C.c_void_p] * 3 + [C.c_int] * 3 + [C.c_void_p]
    _lib.check(L.ntk_gemv_rp_f32(yb.ptr, rp.ptr, xb.ptr, rows, n, dt, None), "gemv_rp_f32")
    y = yb.numpy(np.float32)
    assert (y[rows:rows + 3] == 7.0).all()
    return y[:rows]


@pytest.mark.parametrize("qname", sorted(KQ))
@pytest.mark.parametrize("rows,n", [(1, 256), (16, 512), (17, 1024), (130, 4096), (33, 18432), (20, 32768), (66000, 256)])
def test_rows_and_columns_at_the_edges(qname, rows, n):
    raw, w, x = case(KQ[qname], rows, n, rows + n)
    y = run(raw, KQ[qname], x, rows)
    # (offset and minimum make a weight a difference of two terms of up to twice its largest size)
    big = 2.0 * np.abs(w).reshape(rows, -1, 256).max(2)
    bound = (n / 64 + 40) * 2.0 ** -24 * (big @ np.abs(x.astype(np.float64)).reshape(-1, 256).sum(1))
    assert (np.abs(y - w @ x.astype(np.float64)) <= bound).all()


@pytest.mark.parametrize("qname", sorted(KQ))
@pytest.mark.parametrize("towering", [False, True])
def test_no_further_from_float64_than_the_raw_block_gemv(qname, towering):
    rows, n = 6000, 4096
    raw, w, x = case(KQ[qname], rows, n, 11, towering)
    want = w @ x.astype(np.float64)
    yb = DB(rows * 4)
    ops.launch_gemv(yb, DB.from_numpy(raw), DB.from_numpy(x), rows, n, G.GGML_TO_DT[KQ[qname]])
    err = [np.linalg.norm(y - want) / np.linalg.norm(want) for y in (run(raw, KQ[qname], x, rows), yb.numpy(np.float32)[:rows])]
    print(qname, towering, "repack %.3g raw blocks %.3g" % tuple(err))
    assert err[0] <= 1.03 * err[1]


def test_what_it_refuses():
    L, d = _lib.lib(), DB(1 << 20)
    L.ntk_gemv_rp_f32.argtypes = [C.c_void_p] * 3 + [C.c_int] * 3 + [C.c_void_p]
    q4 = G.GGML_TO_DT[G.GGML_Q4_K]
    for args, code in (((d.ptr, d.ptr, d.ptr, 16, 256, G.GGML_TO_DT[G.GGML_Q8_0]), -1), ((d.ptr, d.ptr, d.ptr, 16, 100, q4), -2), ((d.ptr, d.ptr, d.ptr, 16, 33024, q4), -2),
                       ((d.ptr, d.ptr, None, 16, 256, q4), -5)):
        assert L.ntk_gemv_rp_f32(*args, None) == code


@pytest.mark.parametrize("qname", sorted(KQ))
@pytest.mark.parametrize("kind", ["one sum overflows", "the total overflows", "inf", "nan"])
def test_what_is_not_finite_is_what_the_raw_blocks_give(qname, kind):
    """a sum beyond the range is an infinity of its sign, as from raw blocks (which give NaN for an activation that is not finite)"""
    rows, n, gt = 300, 1024, KQ[qname]
    raw, w, x = case(gt, rows, n, 5)
    blocks = raw.copy().reshape(-1, raw.size // (rows * n // 256))
    at = 208 if qname == "Q6_K" else 0
    blocks[:, at:at + 2] = np.frombuffer(np.float16(30000.0).tobytes(), np.uint8)
    if qname != "Q6_K":
        blocks[:, 2:4] = 0                      # no minima
    raw = blocks.reshape(-1)
    if kind.endswith("overflows"):              # every block alike and every product of one sign: the first super-block's sum alone, or the row's from sums that fit
        raw = np.tile(blocks[:1], (rows * n // 256, 1)).reshape(-1)
        first = G.dequantize(raw, gt, rows * n)[:256].astype(np.float64)
        x = -np.tile(np.sign(first) / np.abs(first).sum(), n // 256)
        x = (np.where(np.arange(n) < 256, 4e39 * x, 0.0) if kind == "one sum overflows" else 2.2e38 * x).astype(np.float32)
    else:
        x[700] = {"inf": np.inf, "nan": np.nan}[kind]
    yb = DB(rows * 4)
    ops.launch_gemv(yb, DB.from_numpy(raw), DB.from_numpy(x), rows, n, G.GGML_TO_DT[gt])
    got, want = run(raw, gt, x, rows), yb.numpy(np.float32)[:rows]
    print(qname, kind, "finite %d inf %d nan %d, raw blocks %d %d %d" % tuple(f(y).sum() for y in (got, want) for f in (np.isfinite, np.isinf, np.isnan)))
    if kind.endswith("overflows"):
        assert np.array_equal(want, np.full(rows, -np.inf, np.float32)) and np.array_equal(got, want)
    else:
        assert not np.isfinite(got).any()
