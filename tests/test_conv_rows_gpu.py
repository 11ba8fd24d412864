"""The short convolution's form of four channels and eight rows a thread (csrc/layer_ops.hip, causal_conv_rows_kernel) against float64: whole and in portions around its
tiles of eight rows and shorter than the history, columns behind the channels, no activation.  Bound as for the general form: 1e-6."""
import numpy as np
import pytest

import fifotar_oracle as O
from test_fifotar_gpu import f32, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("taps", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [4, 36, 1024, 1028])
def test_rows(taps, n):
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(taps + n)
    T = 41
    x, w = f32(g.standard_normal((T, n + 4))), f32(g.standard_normal((n, taps)))
    ref, carried = O.short_conv(x[:, :n].astype(np.float64), w.astype(np.float64))
    for cuts in ([T], [2, 7, 8, 9, 15], [17, 24], [3, 2, 2, 34], [40, 1]):
        parts, st, at = [], None, 0
        for c in cuts:
            o, st = Lr.causal_conv_act(x[at:at + c], w, at, state=st if at else None, n=n)
            parts.append(o)
            at += c
        assert at == T and rel(np.concatenate(parts), ref) < 1e-6, cuts
        if taps > 1:
            assert np.allclose(st, carried, atol=1e-6)
    plain, _ = Lr.causal_conv_act(x, w, 0, act=0, n=n)
    full = np.concatenate([np.zeros((taps - 1, n)), x[:, :n]])
    assert rel(plain, sum(w[:, j] * full[j:j + T] for j in range(taps))) < 1e-6


# as many results as that form is taken for: portions around its tiles, shorter than the history, a last one in the other form
@pytest.mark.parametrize("taps", [1, 2, 3, 4])
@pytest.mark.parametrize("n,T,portions", [(131072, 41, ([41], [7, 8, 9, 17], [24, 17], [40, 1])), (458752, 9, ([9], [2, 3, 4], [5, 2, 2])), (4100, 300, ([300], [230, 70]))])
def test_rows_of_a_million_results(taps, n, T, portions):
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(taps + n)
    x, w = f32(g.standard_normal((T, n + 4))), f32(g.standard_normal((n, taps)))
    ref, carried = O.short_conv(x[:, :n].astype(np.float64), w.astype(np.float64))
    for cuts in portions:
        parts, st, at = [], None, 0
        for c in cuts:
            o, st = Lr.causal_conv_act(x[at:at + c], w, at, state=st if at else None, n=n)
            parts.append(o)
            at += c
        assert at == T and rel(np.concatenate(parts), ref) < 1e-6, cuts
        if taps > 1:
            assert np.allclose(st, carried, atol=1e-6)
