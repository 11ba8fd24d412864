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


@pytest.mark.parametrize("what", ["state", "value"])
def test_values_at_the_end_of_the_range(what):
    """a value between the largest bfloat16 and the largest 32-bit number stays finite in its pieces"""
    from ntransformer_amd import layers as Lr
    T, H, G, dn, dv = 64, 4, 2, 64, 64
    g = np.random.default_rng(3)
    q, k, v, az, wz, rates, bias = _delta_inputs(g, T, H, G, dn, dv)
    state = np.zeros((H, dn, dv))
    top = np.finfo(np.float32).max
    if what == "state":
        state[1, 3, 5] = top * 0.9999
    else:
        v = v * 1e-6
        v.reshape(T, H, dv)[-1, 2, 7] = top * 0.9999
        az[:] = 30.0
    kw = dict(decay_form=Lr.DECAY_EXP_SOFTPLUS, wb=bias, decay_rates=rates, G=G, unit_q=True, unit_k=True, head_gates=True, write_gated=True, q_scale=dn ** -0.5)
    got, st = Lr.gated_recurrence(q, k, v, wz, H, dn, dv, 5, az=az, state=state.astype(np.float32), **kw)
    ref, S = _delta_reference(q, k, v, az, wz, rates, bias, H, G, dn, dv, state.astype(np.float32).astype(np.float64))
    assert np.isfinite(got).all() and np.isfinite(st).all()
    assert np.abs(got - ref.reshape(got.shape)).max() < 1e-5 * max(np.abs(ref).max(), 1e-30)
