"""ntk_gated_delta_step -- a decoded token of the delta rule: convolutions and step in one launch, head norm, silu gate and carried inputs in a second -- against the launches it replaces (ntk_gated_recurrence with the
convolutions inside, ntk_head_rmsnorm_gate) token by token, from an empty state whose memory holds NaN: the state within 1e-6 of its largest value (sums of up to 128 products in float32, in another
order: 16 of the largest one's half ulps), the results within 4e-6 (such a sum over the state, and the head's norm and gate: the difference of a value goes through the norm's factor, up to 3 here), the
carried inputs the same bits.  Sizes below, at and between the rows a lane holds, columns that end inside a wave, one head a group and several."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import layers as Lr
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu


def desc(out, raw, z, state, cw, cst, rates, bias, H, G, dn, dv, pos, taps):
    nqk, na, nz = G * dn, raw.shape[0], z.shape[0]
    bufs = [DB.from_numpy(raw), DB.from_numpy(z)]
    d = Lr.GatedRecurrenceDesc(out.ptr, H * dv, bufs[0].ptr, na, bufs[0].ptr + 4 * nqk, na, bufs[0].ptr + 8 * nqk, na, bufs[1].ptr, nz, bias.ptr, Lr.DECAY_EXP_SOFTPLUS, 1.0,
                               bufs[1].ptr + 4 * H, nz, None, 1e-6, state.ptr, H, dn, dv, dn ** -0.5, pos, 1, None)
    d.G, d.unit_q, d.unit_k, d.head_gates, d.write_gated, d.decay_rates = G, 1, 1, 1, 1, rates.ptr
    d.conv_w, d.conv_state, d.conv_taps = cw.ptr, cst.ptr, taps
    return d, bufs


@pytest.mark.parametrize("H,G,dn,dv,taps", [(16, 8, 128, 128, 4), (4, 2, 24, 40, 4), (3, 3, 13, 7, 2), (2, 2, 65, 100, 1), (4, 1, 64, 64, 3), (1, 1, 32, 16, 4), (6, 3, 33, 128, 4), (16, 1, 8, 5, 4)])
def test_two_launches(H, G, dn, dv, taps):
    L = Lr._bind()
    L.ntk_gated_delta_step.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_float, C.c_void_p]
    g = np.random.default_rng(H * dn + dv)

    def f(*shape):
        return g.standard_normal(shape).astype(np.float32)
    nch = 2 * G * dn + H * dv
    cw, rates, bias = (DB.from_numpy(x) for x in (0.5 * f(nch, taps), np.exp(0.3 * f(H)), 0.2 * f(H)))
    norm = 1.0 + 0.1 * f(dv)
    states = [DB.from_numpy(np.full(H * dn * dv, np.nan, np.float32)) for _ in range(2)]
    carried = [DB.from_numpy(np.full(max(taps - 1, 1) * nch, np.nan, np.float32)) for _ in range(2)]
    nw = DB.from_numpy(norm)
    for pos in range(6):
        raw, z, gate = f(nch), f(2 * H), DB.from_numpy(f(H * dv))
        a, b, c = DB.zeros(H * dv * 4), DB.zeros(H * dv * 4), DB.zeros(H * dv * 4)
        d, keep = desc(a, raw, z, states[0], cw, carried[0], rates, bias, H, G, dn, dv, pos, taps)
        scr = DB.from_numpy(np.full(int(L.ntk_gated_recurrence_scratch_ex(C.byref(d))), np.nan, np.float32))
        d.scratch = scr.ptr
        Lr.check(L.ntk_gated_recurrence(C.byref(d), None), "gated_recurrence")
        Lr.check(L.ntk_head_rmsnorm_gate(b.ptr, H * dv, a.ptr, H * dv, nw.ptr, 0, gate.ptr, H * dv, 2, 1.0, 1, H, dv, 1e-5, None), "head_rmsnorm_gate")
        d, keep2 = desc(c, raw, z, states[1], cw, carried[1], rates, bias, H, G, dn, dv, pos, taps)
        Lr.check(L.ntk_gated_delta_step(C.byref(d), nw.ptr, gate.ptr, 1e-5, None), "gated_delta_step")
        want, got = b.numpy(np.float32), c.numpy(np.float32)
        assert np.isfinite(got).all() and np.abs(got - want).max() <= 4e-6 * max(1.0, np.abs(want).max()), pos
        s0, s1 = (s.numpy(np.float32)[:H * dn * dv] for s in states)
        assert np.abs(s0 - s1).max() <= 1e-6 * max(1.0, np.abs(s0).max())
        if taps > 1:
            assert np.array_equal(carried[0].numpy(np.float32), carried[1].numpy(np.float32))


def test_refused():
    L = Lr._bind()
    L.ntk_gated_delta_step.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_float, C.c_void_p]
    buf = DB.zeros(1 << 20)
    for H, G, dn, dv, taps in [(2, 1, 16, 129, 4), (2, 2, 129, 16, 4), (2, 2, 16, 16, 5), (3, 2, 16, 16, 4)]:
        d, keep = desc(buf, np.zeros(2 * G * dn + H * dv, np.float32), np.zeros(2 * H, np.float32), buf, buf, buf, buf, buf, H, G, dn, dv, 0, taps)
        assert L.ntk_gated_delta_step(C.byref(d), buf.ptr, buf.ptr, 1e-5, None) != 0
