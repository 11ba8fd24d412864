"""The Fifotar family (the scaled form of the layer stack: RMS norms around every sublayer, one residual factor, tied head, capped logits; mixers: attention
over chunks with capped scores, a sink, blended values and an elementwise gate; latent attention with half-split rotation and a per-head gate; the delta rule
with one decay and one write strength per head behind short convolutions; a clipped gated feed-forward) against tests/fifotar_oracle.py -- a float64
restatement that shares nothing with the product.  Every test makes its own small configuration and random bf16-representable weights, writes them as a model
folder and runs them through the C API (the engine's step function, slot cache and state and kernels); the operator tests call include/ntk_layers.h directly.

Error measure: rms of the difference over rms of the reference.  float32 mode is held to 2e-4 (observed ~1e-6), bfloat16 mode to 4e-2."""
import json
import math
import os
import subprocess
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import fifotar_oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL = {"float32": 2e-4, "bfloat16": 4e-2}


def rel(got, ref):
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    return float(np.sqrt(np.mean((got - ref) ** 2)) / (np.sqrt(np.mean(ref ** 2)) + 1e-30))


def row_err(got, ref):
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    return np.sqrt(np.mean((got - ref) ** 2, axis=1)) / np.sqrt(np.mean(ref ** 2))


def make(tmp_path, cfg, seed=1, name="m", gain=1.0):
    w = O.random_weights(cfg, seed, gain)
    folder = str(tmp_path / name)
    O.save_model(folder, cfg, w)
    return folder, w


def engine_for(folder, dtype="float32", ctx=512, slots=1):
    from ntransformer_amd.engine import Engine
    e = Engine()
    e.load_folder(folder, max_context=ctx, dtype=dtype, slots=slots)
    return e


def tokens_for(cfg, n, seed=0):
    return [int(t) for t in np.random.default_rng(seed).integers(0, cfg["vocab"], n)]


def f32(a):
    return np.asarray(a, np.float32)


def mixed(size=24, **kw):
    """attention, delta, latent, delta, attention: both blending layers, both kinds of state, a layer without feed-forward"""
    return O.config([O.attention_layer(size=size), O.delta_layer(), O.latent_layer(scaling={"factor": 4.0, "original": 16, "fast": 4.0, "slow": 1.0}), O.delta_layer(ff=20),
                     O.attention_layer(size=size, heads=4, kv_heads=2)], **kw)


# ====================================================================================================================== operators
@pytest.mark.parametrize("T,n", [(1, 7), (5, 300), (40, 96), (3, 5000), (40, 4500)])
def test_the_seam_owed_result_and_next_norm(T, n):
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(T * n)
    x, y, aw, w = (f32(g.standard_normal(s)) for s in ((T, n), (T, n), (n,), (n,)))
    eps, m = 1e-5, 0.37
    x1 = x + m * O.rms(y.astype(np.float64), aw, eps)
    gx, gh = Lr.rms_seam(x, w, eps, y, aw, m)
    assert rel(gx, x1) < 1e-6 and rel(gh, O.rms(x1, w, eps)) < 1e-6
    gx, gh = Lr.rms_seam(x, w, eps)                                          # nothing owed
    assert np.array_equal(gx, x) and rel(gh, O.rms(x.astype(np.float64), w, eps)) < 1e-6
    gx, gh = Lr.rms_seam(x, None, eps, y, aw, m)                             # nothing follows
    assert gh is None and rel(gx, x1) < 1e-6


@pytest.mark.parametrize("taps", [1, 2, 4, 5, 16])
def test_short_convolution_with_its_carried_inputs(taps):
    """whole, in portions shorter than the history, one token at a time, from a state full of NaN at a sequence's start; extra columns behind the channels"""
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(taps)
    T, n = 23, 37
    x, w = f32(g.standard_normal((T, n + 5))), f32(g.standard_normal((n, taps)))
    ref, carried = O.short_conv(x[:, :n].astype(np.float64), w.astype(np.float64))
    got, st = Lr.causal_conv_act(x, w, 0, n=n)
    assert rel(got, ref) < 1e-6 and rel(st, carried) < 1e-7 if taps > 1 else rel(got, ref) < 1e-6
    for cuts in ([1] * T, [2, 1, 1, 3, 1, 9, 2, 4], [20, 3]):
        parts, st, at = [], None, 0
        for c in cuts:
            o, st = Lr.causal_conv_act(x[at:at + c], w, at, state=st if at else None, n=n)
            parts.append(o)
            at += c
        assert at == T and rel(np.concatenate(parts), ref) < 1e-6, cuts
        if taps > 1:
            assert np.allclose(st, carried, atol=1e-6)
    plain, _ = Lr.causal_conv_act(x, w, 0, act=0, n=n)                      # no activation
    lin = np.zeros((T, n))
    full = np.concatenate([np.zeros((taps - 1, n)), x[:, :n]])
    for j in range(taps):
        lin += w[:, j] * full[j:j + T]
    assert rel(plain, lin) < 1e-6


def test_logit_cap_and_gate_per_head():
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(3)
    x = f32(g.standard_normal((5, 77)) * 40)
    assert rel(Lr.softcap_rows(x, 30.0), 30.0 * np.tanh(x.astype(np.float64) / 30.0)) < 1e-6
    y, gt = f32(g.standard_normal((6, 3 * 11))), f32(g.standard_normal((6, 3)) * 3)
    assert rel(Lr.head_gate(y, gt, 3), (y.reshape(6, 3, 11) * O.sigmoid(gt.astype(np.float64))[:, :, None]).reshape(6, 33)) < 1e-6
    lat, wuv = f32(g.standard_normal((4, 3 * 9))), f32(g.standard_normal((3 * 5, 9)))
    ref = np.einsum("thr,hvr->thv", lat.reshape(4, 3, 9).astype(np.float64), wuv.reshape(3, 5, 9)) * O.sigmoid(gt[:4].astype(np.float64))[:, :, None]
    assert rel(Lr.latent_unfold_value(lat, wuv, 3, gate=gt[:4], head_gate=True), ref.reshape(4, 15)) < 1e-6


@pytest.mark.parametrize("scaling", [None, {"factor": 4.0, "original": 16, "fast": 4.0, "slow": 1.0}, {"factor": 3.0, "original": 256, "fast": 16.0, "slow": 2.0}])
def test_half_split_rotation_into_cache_rows_and_queries(scaling):
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(5)
    R, dr, H, dn, T, pos0 = 10, 12, 3, 6, 9, 1000
    rot = {"base": 10000.0, "dims": dr}
    if scaling:
        rot["scaling"] = scaling
    freq, mag = O.blended_frequencies(rot)
    if scaling:
        assert not np.allclose(freq, O.blended_frequencies({"base": 10000.0, "dims": dr})[0])     # (the ramp does something at these sizes)
    kv, q, nw = f32(g.standard_normal((T, R + dr))), f32(g.standard_normal((T, H * (dn + dr)))), f32(1 + 0.1 * g.standard_normal(R))
    cache, qr = Lr.latent_prepare(kv, nw, 1e-5, R, dr, q, H, freq, mag, dr, pos0, layout=Lr.ROT_HALVES)
    for t in range(T):
        assert rel(cache[pos0 + t, :R], O.rms(kv[t, :R].astype(np.float64), nw, 1e-5)) < 1e-6
        assert rel(cache[pos0 + t, R:], O.rotate_halves(kv[t, R:].astype(np.float64), pos0 + t, freq, mag, dr)) < 1e-5
        for h in range(H):
            v = q[t].reshape(H, dn + dr)[h].astype(np.float64)
            assert rel(qr[t].reshape(H, dn + dr)[h, dn:], O.rotate_halves(v[dn:], pos0 + t, freq, mag, dr)) < 1e-5
            assert np.array_equal(qr[t].reshape(H, dn + dr)[h, :dn], q[t].reshape(H, dn + dr)[h, :dn])
    # the window mixer's rotation takes the layout too
    k, v = f32(g.standard_normal((T, 2 * 8))), f32(g.standard_normal((T, 2 * 3)))
    q2 = f32(g.standard_normal((T, 4 * 8)))
    f8 = np.array([10000.0 ** (-2.0 * i / 8) for i in range(4)])
    cache, qr, _ = Lr.window_prepare_ex(q2, k, v, 4, 2, 8, 3, 50, freq=f8, dims=8, layout=Lr.ROT_HALVES)
    assert rel(cache[50 + 2, :8], O.rotate_halves(k[2, :8].astype(np.float64), 52, f8, 1.0, 8)) < 1e-5
    assert rel(qr[2, 8:16], O.rotate_halves(q2[2, 8:16].astype(np.float64), 52, f8, 1.0, 8)) < 1e-5


def test_values_blended_on_their_way_into_the_cache():
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(6)
    T, H, G, dn, dv = 7, 4, 2, 5, 6
    q, k, v, other = (f32(g.standard_normal(s)) for s in ((T, H * dn), (T, G * dn), (T, G * dv), (T, G * dv)))
    cache, _, kept = Lr.window_prepare_ex(q, k, v, H, G, dn, dv, 3, keep=True)
    assert np.array_equal(kept, v) and np.array_equal(cache[3:, G * dn:], v) and np.array_equal(cache[3:, :G * dn], k)
    cache, _, kept = Lr.window_prepare_ex(q, k, v, H, G, dn, dv, 3, v_other=other, v_blend=0.3)
    assert kept is None and rel(cache[3:, G * dn:], 0.7 * v.astype(np.float64) + 0.3 * other) < 1e-6


def _attention_case(g, H, G, dn, dv, P):
    q = f32(g.standard_normal((P, H * dn)))
    K, V = f32(g.standard_normal((P, G * dn))), f32(g.standard_normal((P, G * dv)))
    return q, K, V, np.concatenate([K, V], axis=1)


@pytest.mark.parametrize("H,G,dn,dv", [(4, 2, 12, 20), (3, 3, 5, 3), (6, 1, 70, 130), (1, 1, 8, 8)])
@pytest.mark.parametrize("pos0,T", [(0, 50), (130, 1), (125, 6), (60, 23)])
@pytest.mark.parametrize("size,cap,sink", [(16, 5.0, True), (64, 0.0, True), (65, 3.0, False), (0, 2.0, True), (1, 0.0, True)])
def test_attention_over_chunks_with_capped_scores_and_a_sink(H, G, dn, dv, pos0, T, size, cap, sink):
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(H * 1000 + pos0 + size)
    P = pos0 + T
    q, K, V, cache = _attention_case(g, H, G, dn, dv, P)
    scale = 2.0 / math.sqrt(dn)
    ref = O.attend(q[pos0:].reshape(T, H, dn).astype(np.float64), K.reshape(P, G, dn).astype(np.float64), V.reshape(P, G, dv).astype(np.float64), pos0, scale,
                   size or None, cap or None, sink).reshape(T, H * dv)
    gate = f32(g.standard_normal((T, H * dv)) * 2)
    for split in (True, False):
        got = Lr.window_attention(q[pos0:], cache, H, G, 1, dn, dv, pos0, size, scale, split=split, chunks=True, softcap=cap, sink=sink)
        assert rel(got, ref) < 1e-5, split
        got = Lr.window_attention(q[pos0:], cache, H, G, 1, dn, dv, pos0, size, scale, split=split, chunks=True, softcap=cap, sink=sink, gate=gate)   # the gate inside the launch
        assert rel(got, ref * O.sigmoid(gate.astype(np.float64))) < 1e-5, split


def test_the_sink_takes_the_weight_when_every_score_is_low():
    """all scores around -30: without the sink the softmax would still hand out weights that sum to one; with it the output all but vanishes"""
    from ntransformer_amd import layers as Lr
    P, dn, dv = 200, 8, 4
    q = f32(np.full((P, dn), 1.0))
    K, V = f32(np.full((P, dn), -30.0 / dn)), f32(np.ones((P, dv)))
    cache = np.concatenate([K, V], axis=1)
    for pos0, T in ((0, P), (P - 1, 1)):
        got = Lr.window_attention(q[pos0:], cache, 1, 1, 1, dn, dv, pos0, 0, 1.0, chunks=True, sink=True)
        n = np.arange(pos0, P) + 1
        want = n * math.exp(-30.0) / (1.0 + n * math.exp(-30.0))
        assert np.allclose(got[:, 0], want, rtol=1e-4, atol=1e-15) and got.max() < 1e-10
        plain = Lr.window_attention(q[pos0:], cache, 1, 1, 1, dn, dv, pos0, 0, 1.0, chunks=True, sink=False)
        assert np.allclose(plain, 1.0, atol=1e-5)


def test_a_towering_key_just_inside_and_just_outside_the_chunk():
    """one key's score stands far above the rest: a query in the same chunk returns that key's value, the first query of the next chunk does not see it --
    for a decoded token and inside a portion, at every place of the chunk's border, with the 64-key steps of the walk falling elsewhere"""
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(8)
    H, G, dn, dv, size, P = 2, 1, 16, 8, 48, 400
    for tower in (0, 47, 48, 95, 96, 143, 335, 336, 383):
        q, K, V, _ = _attention_case(g, H, G, dn, dv, P)
        q *= 0.05
        d = g.standard_normal(dn)
        d /= np.linalg.norm(d)
        K[tower] = 40.0 * d
        q[:, :dn] += 2.0 * d                                                 # head 0 looks for it everywhere; head 1 does not
        cache = np.concatenate([K, V], axis=1)
        last_in = (tower // size) * size + size - 1
        for pos0, T in ((last_in, 1), (last_in + 1, 1), (last_in - 3, 8), (0, min(P, last_in + 30))):
            if pos0 + T > P or pos0 < tower - size:
                continue
            got = Lr.window_attention(q[pos0:pos0 + T], cache[:pos0 + T], H, G, 1, dn, dv, pos0, size, 1.0, chunks=True, sink=True)
            ref = O.attend(q[pos0:pos0 + T].reshape(T, H, dn).astype(np.float64), K[:pos0 + T].reshape(-1, G, dn).astype(np.float64),
                           V[:pos0 + T].reshape(-1, G, dv).astype(np.float64), pos0, 1.0, size, None, True).reshape(T, H * dv)
            assert rel(got, ref) < 1e-5, (tower, pos0, T)
            for t in range(T):
                p = pos0 + t
                if tower <= p <= last_in:
                    assert np.abs(got[t, :dv] - V[tower]).max() < 1e-3, (tower, p)
                elif p == last_in + 1:
                    assert np.abs(got[t, :dv] - V[tower]).max() > 0.05, (tower, p)


def test_a_far_key_among_hundreds_without_a_mask():
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(9)
    H, G, dn, dv, P = 4, 2, 12, 10, 1300
    for tower in (0, 63, 64, 700, 1279):
        q, K, V, _ = _attention_case(g, H, G, dn, dv, P)
        q *= 0.05
        d = g.standard_normal(dn)
        d /= np.linalg.norm(d)
        K[tower, dn:] = 40.0 * d                                             # key head 1
        q[-1, 2 * dn:3 * dn] += 2.0 * d                                      # query head 2 reads key head 1
        cache = np.concatenate([K, V], axis=1)
        for split in (True, False):
            got = Lr.window_attention(q[-1:], cache, H, G, 1, dn, dv, P - 1, 0, 1.0, split=split, chunks=True, softcap=60.0, sink=True)
            assert np.abs(got[0, 2 * dv:3 * dv] - V[tower, dv:]).max() < 1e-3, (tower, split)


def _delta_inputs(g, T, H, G, dn, dv):
    q, k = f32(g.standard_normal((T, G * dn))), f32(g.standard_normal((T, G * dn)))
    v = f32(g.standard_normal((T, H * dv)))
    az, wz = f32(g.standard_normal((T, H)) * 2), f32(g.standard_normal((T, H)))
    rates, bias = f32(np.exp(g.uniform(-3, 0.5, H))), f32(g.uniform(-2, 1, H))
    return q, k, v, az, wz, rates, bias


def _delta_reference(q, k, v, az, wz, rates, bias, H, G, dn, dv, state=None):
    T = q.shape[0]
    share = np.arange(H) // (H // G)
    qq = (O.unit(q.reshape(T, G, dn).astype(np.float64)) * dn ** -0.5)[:, share]
    kk = O.unit(k.reshape(T, G, dn).astype(np.float64))[:, share]
    decay = np.exp(-rates.astype(np.float64) * O.softplus(wz.astype(np.float64) + bias))
    return O.delta_walk(qq, kk, v.reshape(T, H, dv).astype(np.float64), O.sigmoid(az.astype(np.float64)), decay, state)


DELTA_SHAPES = [(1, 1, 1, 1), (4, 2, 8, 8), (6, 3, 32, 64), (3, 3, 13, 7), (2, 1, 70, 130), (2, 2, 128, 96), (1, 1, 200, 24)]


@pytest.mark.parametrize("H,G,dn,dv", DELTA_SHAPES)
def test_delta_rule_with_per_head_gates_whole_in_portions_and_token_by_token(H, G, dn, dv):
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(H * 100 + dn)
    T = 45
    q, k, v, az, wz, rates, bias = _delta_inputs(g, T, H, G, dn, dv)
    ref, S = _delta_reference(q, k, v, az, wz, rates, bias, H, G, dn, dv)
    kw = dict(decay_form=Lr.DECAY_EXP_SOFTPLUS, wb=bias, decay_rates=rates, G=G, unit_q=True, unit_k=True, head_gates=True, write_gated=True, q_scale=dn ** -0.5)
    got, st = Lr.gated_recurrence(q, k, v, wz, H, dn, dv, 0, az=az, **kw)                      # (the state starts full of NaN: position 0 must not read it)
    assert rel(got, ref.reshape(T, H * dv)) < 1e-5 and rel(st, S) < 1e-5
    for cuts in ([1] * T, [2, 9, 3, 8, 1, 17, 5], [44, 1]):
        parts, st, at = [], None, 0
        for c in cuts:
            o, st = Lr.gated_recurrence(q[at:at + c], k[at:at + c], v[at:at + c], wz[at:at + c], H, dn, dv, at, az=az[at:at + c], state=st, **kw)
            parts.append(o)
            at += c
        assert at == T and rel(np.concatenate(parts), ref.reshape(T, H * dv)) < 1e-5 and rel(st, S) < 1e-5, cuts


@pytest.mark.parametrize("H,G,dn,dv", [(4, 2, 32, 64), (2, 2, 128, 128), (3, 1, 9, 11)])
def test_delta_rule_long_portions_walked_in_segments(H, G, dn, dv):
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(dn)
    T = 700
    q, k, v, az, wz, rates, bias = _delta_inputs(g, T, H, G, dn, dv)
    ref, S = _delta_reference(q, k, v, az, wz, rates, bias, H, G, dn, dv)
    kw = dict(decay_form=Lr.DECAY_EXP_SOFTPLUS, wb=bias, decay_rates=rates, G=G, unit_q=True, unit_k=True, head_gates=True, write_gated=True, q_scale=dn ** -0.5)
    got, st = Lr.gated_recurrence(q, k, v, wz, H, dn, dv, 0, az=az, **kw)
    assert rel(got, ref.reshape(T, H * dv)) < 1e-4 and rel(st, S) < 1e-4
    a, st = Lr.gated_recurrence(q[:130], k[:130], v[:130], wz[:130], H, dn, dv, 0, az=az[:130], **kw)
    b, st = Lr.gated_recurrence(q[130:], k[130:], v[130:], wz[130:], H, dn, dv, 130, az=az[130:], state=st, **kw)
    assert rel(np.concatenate([a, b]), ref.reshape(T, H * dv)) < 1e-4 and rel(st, S) < 1e-4


@pytest.mark.parametrize("H,G,dn,dv,T", [(1, 1, 64, 16, 32), (4, 2, 64, 48, 33), (2, 2, 128, 128, 63), (6, 3, 128, 16, 64), (2, 1, 128, 144, 65), (16, 16, 128, 128, 513)])
def test_delta_rule_in_chunks_on_the_matrix_instructions(H, G, dn, dv, T):
    """one chunk, partial last chunks, both widths; strong decay (products that underflow) and none; a portion behind a state; and what comes before a NaN stays clean"""
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(T + dn)
    q, k, v, az, wz, rates, bias = _delta_inputs(g, T + 40, H, G, dn, dv)
    for scale in (1.0, 60.0, 0.0):
        r = (rates * scale).astype(np.float32)
        ref, S = _delta_reference(q, k, v, az, wz, r, bias, H, G, dn, dv)
        ref = ref.reshape(T + 40, H * dv)
        kw = dict(decay_form=Lr.DECAY_EXP_SOFTPLUS, wb=bias, decay_rates=r, G=G, unit_q=True, unit_k=True, head_gates=True, write_gated=True, q_scale=dn ** -0.5)
        a, st = Lr.gated_recurrence(q[:T], k[:T], v[:T], wz[:T], H, dn, dv, 0, az=az[:T], **kw)
        b, st = Lr.gated_recurrence(q[T:], k[T:], v[T:], wz[T:], H, dn, dv, T, az=az[T:], state=st, **kw)
        # 32-bit sums of 128 + 32 terms per token; the state keeps what a token left for as long as the decay lets it: the bound of the walk at 45 tokens
        assert rel(np.concatenate([a, b]), ref) < 1e-5 and rel(st, S) < 1e-5, scale
    at = T - 7
    v[at] = np.nan
    a, st = Lr.gated_recurrence(q[:T], k[:T], v[:T], wz[:T], H, dn, dv, 0, az=az[:T], **kw)
    assert rel(a[:at], ref[:at]) < 1e-5 and np.isnan(a[at:]).all() and np.isnan(st).all()


@pytest.mark.parametrize("H,G,dn,dv,T", [(2, 1, 64, 48, 47), (2, 1, 64, 48, 48), (3, 3, 128, 128, 49), (2, 2, 128, 144, 63), (2, 2, 128, 144, 64), (1, 1, 64, 256, 97)])
def test_delta_rule_where_chunks_take_over_from_the_walk(H, G, dn, dv, T):
    """portions around the length from which the chunks are taken, for values up to 128 and wider, against the reference and behind a state"""
    test_delta_rule_in_chunks_on_the_matrix_instructions(H, G, dn, dv, T)


@pytest.mark.parametrize("H,G,dn,dv,taps", [(4, 2, 8, 8, 4), (6, 3, 32, 64, 4), (3, 3, 13, 7, 2), (2, 1, 70, 130, 5), (5, 1, 16, 300, 1), (2, 2, 128, 96, 16)])
def test_decoded_tokens_pass_their_convolutions_inside_the_recurrence(H, G, dn, dv, taps):
    """raw q, k, v of one token at a time, the short convolutions inside the pre-pass's launch: the same outputs, state and carried inputs as the convolution as an
    operator of its own in front of a whole portion; a sequence may change from one form to the other at any token"""
    from ntransformer_amd import layers as Lr
    g = np.random.default_rng(H * 100 + dn + taps)
    T = 21
    q, k, v, az, wz, rates, bias = _delta_inputs(g, T, H, G, dn, dv)
    cw = f32(g.standard_normal((2 * G * dn + H * dv, taps)) * 0.5)
    raw = np.concatenate([q, k, v], axis=1)
    conv, carried = O.short_conv(raw.astype(np.float64), cw.astype(np.float64))
    cq, ck, cv = f32(conv[:, :G * dn]), f32(conv[:, G * dn:2 * G * dn]), f32(conv[:, 2 * G * dn:])
    ref, S = _delta_reference(cq, ck, cv, az, wz, rates, bias, H, G, dn, dv)
    kw = dict(decay_form=Lr.DECAY_EXP_SOFTPLUS, wb=bias, decay_rates=rates, G=G, unit_q=True, unit_k=True, head_gates=True, write_gated=True, q_scale=dn ** -0.5)
    for first in (0, 9):                                                     # the first tokens as one portion through the operators, the rest token by token
        outs, st, cst = [], None, None
        if first:
            conv_a, cst = Lr.causal_conv_act(raw[:first], cw, 0)
            o, st = Lr.gated_recurrence(conv_a[:, :G * dn], conv_a[:, G * dn:2 * G * dn], conv_a[:, 2 * G * dn:], wz[:first], H, dn, dv, 0, az=az[:first], **kw)
            outs.append(o)
        for t in range(first, T):
            o, st, cst = Lr.gated_recurrence(q[t:t + 1], k[t:t + 1], v[t:t + 1], wz[t:t + 1], H, dn, dv, t, az=az[t:t + 1], state=st, conv_w=cw, conv_state=cst, **kw)
            outs.append(o)
        assert rel(np.concatenate(outs), ref.reshape(T, H * dv)) < 1e-5 and rel(st, S) < 1e-5, first
        if taps > 1:
            assert np.allclose(cst, carried, atol=1e-6)


def test_the_delta_rule_replaces_what_a_key_held_and_remembers_it_without_decay():
    """decay one (a large negative pre-activation), write strength one: a key written at token 0 is read back 600 tokens later; writing the SAME key again
    replaces its value instead of adding to it -- plain linear attention would return the sum"""
    from ntransformer_amd import layers as Lr
    T, dn, dv = 650, 16, 8
    g = np.random.default_rng(10)
    e0, e1 = np.eye(dn)[0], np.eye(dn)[1]
    k = f32(np.tile(e1, (T, 1)) * 1e-4)                                      # (a key of length 1e-4 along e1 still has the unit e1: it rewrites e1's slot only)
    q = f32(np.tile(e0, (T, 1)))
    v = f32(g.standard_normal((T, dv)))
    k[0], k[300] = 3.0 * e0, 0.5 * e0
    az, wz = f32(np.full((T, 1), 40.0)), f32(np.full((T, 1), -60.0))
    kw = dict(decay_form=Lr.DECAY_EXP_SOFTPLUS, decay_param=1.0, G=1, unit_q=True, unit_k=True, head_gates=True, write_gated=True, q_scale=1.0, unit_eps=1e-20)
    out, _ = Lr.gated_recurrence(q, k, v, wz, 1, dn, dv, 0, az=az, **kw)
    assert np.abs(out[:300] - v[0]).max() < 1e-4 and np.abs(out[300:] - v[300]).max() < 1e-4
    parts, st = [], None
    for at in range(0, T, 97):
        o, st = Lr.gated_recurrence(q[at:at + 97], k[at:at + 97], v[at:at + 97], wz[at:at + 97], 1, dn, dv, at, az=az[at:at + 97], state=st, **kw)
        parts.append(o)
    assert np.abs(np.concatenate(parts) - out).max() < 1e-5
    wz2 = wz.copy()
    wz2[100] = 0.0                                                           # one token forgets: softplus(0) = ln 2, the state halves once
    out2, _ = Lr.gated_recurrence(q, k, v, wz2, 1, dn, dv, 0, az=az, **kw)
    assert np.abs(out2[100:300] - 0.5 * v[0]).max() < 1e-4 and np.abs(out2[:100] - v[0]).max() < 1e-4


# ====================================================================================================================== whole models
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_whole_prompt_with_the_stream_after_every_layer(tmp_path, dtype):
    cfg = mixed()
    folder, w = make(tmp_path, cfg, seed=2)
    toks = tokens_for(cfg, 60, seed=3)
    streams = []
    ref, _ = O.forward(cfg, w, toks, layers_out=streams)
    e = engine_for(folder, dtype)
    assert e.layer_runs == 5
    e.seq_capture(True)
    s = e.seq_acquire()
    got = e.seq_forward(s, toks)
    cap = e.seq_captured(len(toks))
    for i in range(5):
        assert rel(cap[i], streams[i]) < TOL[dtype], i
    assert rel(got, ref) < TOL[dtype]
    e.seq_capture(False)
    e.seq_release(s)
    s = e.seq_acquire()
    some = e.seq_forward(s, toks, want=[0, 7, 59])                           # wanted places only
    assert rel(some, ref[[0, 7, 59]]) < TOL[dtype]
    e.close()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_prefill_against_token_by_token_and_portions(tmp_path, dtype):
    """the same sequence whole, one token at a time and in portions down to two tokens: same logits at every position.  150 tokens in chunks of 24: portions
    start and end on both sides of the chunk edges, of the attention's 64-key steps, of the convolution's reach, of the recurrence's token batches and of the
    switch between the few-row and the tiled products"""
    cfg = mixed()
    folder, w = make(tmp_path, cfg, seed=3)
    e = engine_for(folder, dtype)
    toks = tokens_for(cfg, 150, seed=4)
    ref, _ = O.forward(cfg, w, toks)
    s = e.seq_acquire()
    whole = e.seq_forward(s, toks)
    e.seq_release(s)
    assert rel(whole, ref) < TOL[dtype] and row_err(whole, ref).max() < 3 * TOL[dtype]
    s = e.seq_acquire()
    one = np.concatenate([e.seq_forward(s, toks[i:i + 1]) for i in range(len(toks))])
    e.seq_release(s)
    assert rel(one, ref) < TOL[dtype] and row_err(one, ref).max() < 3 * TOL[dtype]
    for cuts in ([2, 9, 3, 8, 17, 2, 30, 1, 5, 64, 2, 7], [23, 2, 2, 2, 19, 48, 1, 1, 1, 24, 27], [2] * 75):
        s = e.seq_acquire()
        parts, at = [], 0
        for n in cuts:
            parts.append(e.seq_forward(s, toks[at:at + n]))
            at += n
        assert at == len(toks) and e.seq_length(s) == at
        cut = np.concatenate(parts)
        e.seq_release(s)
        assert rel(cut, ref) < TOL[dtype] and row_err(cut, ref).max() < 3 * TOL[dtype], cuts
        if dtype == "float32":
            assert rel(one, whole) < 1e-5 and rel(cut, whole) < 1e-5
    e.close()


def test_first_tokens_of_a_sequence(tmp_path):
    cfg = mixed()
    folder, w = make(tmp_path, cfg, seed=5)
    e = engine_for(folder)
    for n in (1, 2, 3, 4, 5):
        toks = tokens_for(cfg, n, seed=n)
        s = e.seq_acquire()
        assert rel(e.seq_forward(s, toks), O.forward(cfg, w, toks)[0]) < TOL["float32"]
        e.seq_release(s)
    e.close()


def test_two_slots_side_by_side_and_a_slot_used_again(tmp_path):
    """two sequences advance in turn, each alone would give the same; a freed slot (cache rows, state and convolution inputs of a longer sequence still there) is
    taken by a shorter one; a sequence with recurrent state can be cut back to its start only"""
    cfg = mixed()
    folder, w = make(tmp_path, cfg, seed=6)
    e = engine_for(folder, slots=2)
    ta, tb = tokens_for(cfg, 60, 1), tokens_for(cfg, 33, 2)
    ra, rb = O.forward(cfg, w, ta)[0], O.forward(cfg, w, tb)[0]
    a, b = e.seq_acquire(), e.seq_acquire()
    assert a != b
    with pytest.raises(Exception):
        e.seq_acquire()
    got_a, got_b = [], []
    cuts_a, cuts_b = [20, 1, 1, 30, 8], [2, 1, 25, 5]
    ia = ib = 0
    for k in range(5):
        got_a.append(e.seq_forward(a, ta[ia:ia + cuts_a[k]])); ia += cuts_a[k]
        if k < 4:
            got_b.append(e.seq_forward(b, tb[ib:ib + cuts_b[k]])); ib += cuts_b[k]
    assert rel(np.concatenate(got_a), ra) < TOL["float32"] and rel(np.concatenate(got_b), rb) < TOL["float32"]
    e.seq_release(a)
    c = e.seq_acquire()
    assert c == a
    tc = tokens_for(cfg, 9, 3)
    assert rel(e.seq_forward(c, tc), O.forward(cfg, w, tc)[0]) < TOL["float32"]
    with pytest.raises(Exception):
        e.seq_truncate(c, 4)
    e.seq_truncate(c, 0)
    assert rel(e.seq_forward(c, tb[:5]), rb[:5]) < TOL["float32"]
    e.close()


def _other():
    A, D, Lt = O.attention_layer, O.delta_layer, O.latent_layer
    return {
        "one of everything": O.config([A(heads=1, kv_heads=1, dim=1, vdim=1, size=1, ff=1), D(heads=1, kv_heads=1, dim=1, vdim=1, conv=1, ff=1),
                                       Lt(heads=1, dim=1, rot_dim=2, vdim=1, kv_rank=1, q_rank=1, ff=1)], vocab=5, width=8),
        "all sizes equal, factors one": O.config([D(heads=4, kv_heads=4, dim=16, vdim=16, conv=2, ff=16), A(heads=4, kv_heads=4, dim=16, vdim=16, size=16, ff=16, scale=1.0),
                                                  Lt(heads=4, dim=16, rot_dim=16, vdim=16, kv_rank=16, q_rank=16, ff=16, scale=1.0), A(heads=4, kv_heads=4, dim=16, vdim=16, size=16, ff=16)],
                                                 vocab=16, width=16, mult=1.0, embed_scale=1.0),
        "multiples of nothing": O.config([Lt(heads=3, dim=7, rot_dim=6, vdim=5, kv_rank=11, q_rank=13, ff=29), D(heads=6, kv_heads=2, dim=13, vdim=7, conv=3, ff=17),
                                          A(heads=3, kv_heads=1, dim=7, vdim=5, size=19, ff=29), A(heads=6, kv_heads=1, dim=9, vdim=5, size=7, ff=0)], vocab=31, width=23, mult=0.3),
        "wide heads": O.config([A(heads=2, kv_heads=1, dim=96, vdim=136, size=40, ff=40), D(heads=2, kv_heads=1, dim=140, vdim=72, conv=4, ff=0),
                                Lt(heads=2, dim=72, rot_dim=40, vdim=130, kv_rank=136, q_rank=48, ff=40)], vocab=50, width=64),
        "nothing but recurrences without feed-forward": O.config([D(), D(heads=2, kv_heads=2, conv=5)]),
        "no mask, no caps, no blending": O.config([A(size=0, softcap=0.0, v_mix=False), A(size=0, softcap=0.0, v_mix=False), Lt()], logit_softcap=0.0),
        "one blending layer among others": O.config([A(v_mix=False, size=10), D(), A(v_mix=True, size=20), A(v_mix=False, size=30)]),
        "blending layers apart": O.config([D(), A(heads=2, kv_heads=2, dim=4, vdim=12, size=33), Lt(), A(heads=6, kv_heads=2, dim=8, vdim=12, size=9), D(ff=12), A(heads=4, kv_heads=2, dim=5, vdim=12, size=0)]),
        "a tight clamp": O.config([A(limit=0.05), D(ff=16, limit=0.05)]),
    }


OTHER = _other()


# Heads of ONE value: the norm behind a sublayer divides a single number by its own magnitude, and a sum that nearly cancels comes out of it as large as any
# other -- what the few-row and the tiled forms round differently in the last bit is then a visible difference.  That configuration is held to 50 x the
# tolerance where it decodes (observed: 5e-3 on one token in 70; its whole prompt is as exact as the others').
LOOSE = {"one of everything": 50.0}


@pytest.mark.parametrize("name", sorted(OTHER))
def test_other_sizes(tmp_path, name):
    cfg = OTHER[name]
    folder, w = make(tmp_path, cfg, seed=7)
    toks = tokens_for(cfg, 70, seed=8)
    streams = []
    ref, _ = O.forward(cfg, w, toks, layers_out=streams)
    for dtype in ("float32", "bfloat16"):
        e = engine_for(folder, dtype)
        e.seq_capture(True)
        s = e.seq_acquire()
        got = e.seq_forward(s, toks[:61])
        assert rel(e.seq_captured(61)[-1], streams[-1][:61]) < TOL[dtype], dtype
        e.seq_capture(False)
        tail = np.concatenate([e.seq_forward(s, toks[61:63])] + [e.seq_forward(s, [t]) for t in toks[63:]])
        assert rel(got, ref[:61]) < TOL[dtype], dtype
        assert rel(np.concatenate([got, tail]), ref) < TOL[dtype] * LOOSE.get(name, 1.0), dtype
        e.close()


def test_long_decoding_and_a_prompt_longer_than_one_internal_pass(tmp_path):
    """1100 tokens in one internal pass (beyond one: test_long_portions_gpu.py); then 200 tokens one by one across several chunk edges, the convolutions and the state carried"""
    cfg = O.config([O.attention_layer(size=88), O.delta_layer(), O.attention_layer(size=200), O.latent_layer(ff=0)])
    folder, w = make(tmp_path, cfg, seed=9)
    toks = tokens_for(cfg, 1100, seed=10)
    e = engine_for(folder, ctx=1300)
    s = e.seq_acquire()
    got = e.seq_forward(s, toks, want=[0, 1023, 1024, 1099])
    ref, _ = O.forward(cfg, w, toks)
    assert rel(got, ref[[0, 1023, 1024, 1099]]) < TOL["float32"]
    e.seq_release(s)
    s = e.seq_acquire()
    e.seq_forward(s, toks[:900], want=[])
    dec = np.concatenate([e.seq_forward(s, [t]) for t in toks[900:]])
    assert rel(dec, ref[900:]) < TOL["float32"] and row_err(dec, ref[900:]).max() < 3 * TOL["float32"]
    with pytest.raises(Exception):                                          # the slot's positions are used up
        e.seq_forward(s, toks[:300])
    e.close()


def test_greedy_generation_through_the_engine_and_the_command_line(tmp_path):
    cfg = mixed()
    folder, w = make(tmp_path, cfg, seed=15, gain=2.0)
    prompt = tokens_for(cfg, 12, seed=16)
    want = O.greedy(cfg, w, prompt, 10)
    e = engine_for(folder)
    assert e.is_sequence_model and e.vocab_size == cfg["vocab"] and e.hidden_size == cfg["width"] and e.n_layers == 5
    assert e.generate_tokens(prompt, 10, temperature=0.0, stop_at_eos=False) == want
    assert e.generate_tokens(prompt, 10, temperature=0.0, stop_at_eos=False) == want      # the slot came back, its old state is not read
    a = e.generate_tokens(prompt, 8, temperature=0.9, top_k=20, top_p=0.95, seed=5, stop_at_eos=False)
    assert a == e.generate_tokens(prompt, 8, temperature=0.9, top_k=20, top_p=0.95, seed=5, stop_at_eos=False) and len(a) == 8
    assert rel(e.forward(prompt[:8], 0), O.forward(cfg, w, prompt[:8])[0][-1]) < TOL["float32"]
    assert rel(e.forward(prompt[8:], 8), O.forward(cfg, w, prompt)[0][-1]) < TOL["float32"]
    e.close()
    cli = os.path.join(ROOT, "ntransformer_amd", "ntransformer")
    r = subprocess.run([cli, "-m", folder, "--dtype", "float32", "--tokens", ",".join(map(str, prompt)), "-n", "10", "-t", "0", "--repeat-penalty", "1"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [int(t) for t in r.stdout.strip().splitlines()[-1].split(",")] == want


def test_trace_runner_replays_steps(tmp_path):
    cfg = mixed()
    folder, w = make(tmp_path, cfg, seed=17)
    ta, tb = tokens_for(cfg, 40, 1), tokens_for(cfg, 6, 2)
    ra, rb = O.forward(cfg, w, ta)[0], O.forward(cfg, w, tb)[0]
    steps = [
        {"step": 0, "entries": [{"id": "a", "tokens": ta[:23], "want": [0, 22]}], "end": []},
        {"step": 1, "entries": [{"id": "a", "tokens": ta[23:25], "want": []}], "end": []},
        {"step": 2, "entries": [{"id": "a", "tokens": ta[25:], "want": [14]}], "end": ["a"]},
        {"step": 3, "entries": [{"id": "b", "tokens": tb, "want": [5]}], "end": ["b"]},
    ]
    V = cfg["vocab"]
    for dtype in ("float32", "bfloat16"):
        out = tmp_path / ("out_" + dtype)
        out.mkdir()
        r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", folder, "--dtype", dtype, "--out", str(out), "--max-tokens", "40"],
                           input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, r.stderr[-2000:]
        assert [l for l in r.stdout.splitlines() if l.startswith("done")] == ["done %d" % k for k in range(4)]
        assert not (out / "1.f32").exists()
        assert rel(np.fromfile(out / "0.f32", np.float32).reshape(-1, V), ra[[0, 22]]) < TOL[dtype]
        assert rel(np.fromfile(out / "2.f32", np.float32).reshape(-1, V), ra[[39]]) < TOL[dtype]
        assert rel(np.fromfile(out / "3.f32", np.float32).reshape(-1, V), rb[[5]]) < TOL[dtype]


@pytest.mark.parametrize("bad", ["mixer type", "tensor", "kv_heads", "kind", "blend sizes", "taps"])
def test_refused_folders(tmp_path, bad):
    from ntransformer_amd.engine import Engine
    cfg = mixed()
    w = O.random_weights(cfg, 1)
    if bad == "mixer type": cfg["layers"][1]["type"] = "lightning"
    elif bad == "tensor": del w["l1.mix.A_log"]
    elif bad == "kv_heads": cfg["layers"][1]["mixer"]["kv_heads"] = 3
    elif bad == "kind": cfg["layers"][0]["mlp"]["kind"] = "moe"
    elif bad == "blend sizes": cfg["layers"][4]["mixer"]["kv_heads"] = 1
    else: cfg["layers"][3]["mixer"]["conv"] = 3
    folder = str(tmp_path / "bad")
    O.save_model(folder, cfg, w)
    e = Engine()
    with pytest.raises(Exception):
        e.load_folder(folder, max_context=64, dtype="float32")
    e.close()


_COUNT_ROUNDINGS = """
import sys
sys.path.insert(0, {root!r}); sys.path.insert(0, {tests!r})
import torch
from torch.profiler import profile, ProfilerActivity
import test_fifotar_gpu as T
e = T.engine_for({folder!r}, "bfloat16")
for turn in range(2):
    s = e.seq_acquire()
    if turn == 0: e.seq_forward(s, {toks!r})
    else:
        with profile(activities=[ProfilerActivity.CUDA]) as p:
            e.seq_forward(s, {toks!r})
            torch.cuda.synchronize()
    e.seq_release(s)
names = [ev.name for ev in p.events()]
print("LAUNCHES", sum("ntk::" in n for n in names), "ROUNDINGS", sum("round_rows_kernel" in n for n in names))
"""


@pytest.mark.parametrize("ff,width", [(96, 64), (112, 64), (128, 64)])
def test_rows_are_rounded_only_for_units_whose_two_products_take_them(tmp_path, ff, width):
    """a feed-forward size that is no multiple of 64: its down product reads 32-bit rows, so the unit's input is not rounded in a launch of its own either"""
    cfg = O.config([O.attention_layer(ff=ff), O.delta_layer(ff=ff), O.latent_layer(ff=ff)], width=width)
    folder, w = make(tmp_path, cfg)
    toks = tokens_for(cfg, 40)
    here = os.path.dirname(os.path.abspath(__file__))
    code = _COUNT_ROUNDINGS.format(root=os.path.dirname(here), tests=here, folder=folder, toks=toks)
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    launches, roundings = (int(x) for x in out.stdout.split("LAUNCHES")[1].split("ROUNDINGS"))
    assert launches > 20 and roundings == 0
    e = engine_for(folder, "bfloat16")
    assert rel(e.seq_forward(e.seq_acquire(), toks), O.forward(cfg, w, toks)[0]) < TOL["bfloat16"]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("ff,width,T", [(2816, 192, 40), (2816, 192, 130), (1408, 192, 300)])
def test_wide_units_leave_their_activations_in_the_first_products_launch(tmp_path, dtype, ff, width, T):
    """sizes for which a unit's first product takes the direct form (in bfloat16 its input and its activations are rounded rows): the other tests' units are too narrow for it"""
    import ctypes as C
    from ntransformer_amd import _lib
    f = _lib.lib().ntk_dense_unit_direct
    f.argtypes, f.restype = [C.c_int] * 7 + [C.c_size_t], C.c_int
    assert f(9 if dtype == "bfloat16" else 0, T, 1, T, width, ff, 0, 1 << 24) == 1
    cfg = O.config([O.attention_layer(ff=ff), O.delta_layer(ff=ff), O.latent_layer(ff=ff)], width=width)
    folder, w = make(tmp_path, cfg, seed=4)
    toks = tokens_for(cfg, T)
    e = engine_for(folder, dtype)
    assert rel(e.seq_forward(e.seq_acquire(), toks), O.forward(cfg, w, toks)[0]) < TOL[dtype]
