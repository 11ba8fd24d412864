"""The delta rule in chunks (csrc/delta_chunk.hip.h) takes 32-bit values apart into three bfloat16 pieces: values near both ends of the range, lengths around a chunk's and
two chunks' edges, both widths, behind a state, against float64.  Bound: 1e-6 of the result's norm, four times what 32-bit sums of this length leave."""
import numpy as np
import pytest

from test_fifotar_gpu import _delta_inputs, _delta_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dn", [64, 128])
@pytest.mark.parametrize("T", [48, 63, 64, 65, 97])
@pytest.mark.parametrize("size", [1e-30, 1.0, 1e30])
def test_sizes_of_values(dn, T, size):
    from ntransformer_amd import layers as Lr
    H, G, dv = 4, 2, 64
    g = np.random.default_rng(T + dn)
    q, k, v, az, wz, rates, bias = _delta_inputs(g, T, H, G, dn, dv)
    v = (v * size).astype(np.float32)
    state = (g.standard_normal((H, dn, dv)) * size).astype(np.float32)
    kw = dict(decay_form=Lr.DECAY_EXP_SOFTPLUS, wb=bias, decay_rates=rates, G=G, unit_q=True, unit_k=True, head_gates=True, write_gated=True, q_scale=dn ** -0.5)
    got, st = Lr.gated_recurrence(q, k, v, wz, H, dn, dv, 5, az=az, state=state, **kw)
    ref, S = _delta_reference(q, k, v, az, wz, rates, bias, H, G, dn, dv, state.astype(np.float64))
    assert np.linalg.norm((got - ref.reshape(got.shape)) / size) < 1e-6 * np.linalg.norm(ref / size)
    assert np.linalg.norm((st.reshape(S.shape) - S) / size) < 1e-6 * np.linalg.norm(S / size)
