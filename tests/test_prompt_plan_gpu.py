"""The FP16 product of prompts of 321 to about 900 tokens, two chunks a workgroup with K in two or four, against the same tokens 64 at a time (one chunk, K in other pieces)."""
import numpy as np
import pytest

from ntransformer_amd import gguf as G, ops
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu


# chunks six and seven (an odd one beside its pair) and eleven, K of whole and uneven trips, rows past the last tile
@pytest.mark.parametrize("fmt", ["Q8_0", "Q4_0", "Q4_K"])
@pytest.mark.parametrize("T,rows,K", [(321, 4096, 4096), (400, 4096, 1792), (449, 6160, 2048), (700, 4096, 2304)])
def test_wide_plans(fmt, T, rows, K):
    gt = getattr(G, "GGML_" + fmt)
    dt, g = G.GGML_TO_DT[gt], np.random.default_rng(T + K)
    W = DB.from_numpy(np.frombuffer(G.synth_tensor(g, gt, rows, K), np.uint8))
    x = g.standard_normal((T, K)).astype(np.float32)
    y = DB.zeros(T * rows * 4)
    assert ops.gemm_quant_ws(y, W, DB.from_numpy(x), T, rows, K, dt) == 0
    got = y.numpy(np.float32).reshape(T, rows)
    for t in range(0, T, 64):
        n = min(64, T - t)
        part = DB.zeros(n * rows * 4)
        assert ops.gemm_quant_ws(part, W, DB.from_numpy(x[t:t + n]), n, rows, K, dt) == 0
        want = part.numpy(np.float32).reshape(n, rows)
        # both are sums of K / 32 block products in pieces: 2^-24 (K / 32 + 4) of sqrt(K / 32) of the result's size at the very most, 1.5e-5 at 4096 columns
        assert np.isfinite(got).all() and np.abs(got[t:t + n] - want).max() <= 1.5e-5 * np.abs(want).max()
