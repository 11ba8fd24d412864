"""The matrix-instruction form of the prompt attention (csrc/attention_tile.hip.h) at the edges of its tiles (32 rows, 32 keys, head sizes below, at and between its operand
sizes) against float64: every option of the window mixer that it takes, and the latent mixer's two-part keys.  Bound on a result: scores are off by (dk + 4) * 2^-24 of
sum |q k| (at most ~30 here), weights by that and an exponential's rounding, the weighted sum by its (keys + 4) additions: 2e-5 of the largest value."""
import numpy as np
import pytest

from ntransformer_amd import layers as Lr

pytestmark = pytest.mark.gpu


def reference(q, k, v, pos0, scale, window=0, chunks=False, keep=0, cap=0.0, sinks=None, slopes=None):
    T, H, _ = q.shape
    G = k.shape[1]
    out = np.zeros((T, H, v.shape[2]))
    j = np.arange(k.shape[0])
    for t in range(T):
        p = pos0 + t
        vis = j <= p
        if window:
            vis &= ((j // window == p // window) if chunks else (p - j < window)) | (j < keep)
        for h in range(H):
            s = (k[:, h // (H // G)] @ q[t, h]) * scale
            if slopes is not None:
                s = s - slopes[h] * (p - j)
            if cap:
                s = cap * np.tanh(s / cap)
            s = np.where(vis, s, -np.inf)
            m = s.max() if sinks is None else max(s.max(), sinks[h])
            e = np.exp(s - m)
            out[t, h] = (e / (e.sum() + (0.0 if sinks is None else np.exp(sinks[h] - m)))) @ v[:, h // (H // G)]
    return out


def values(T, pos0, H, G, dn, dv, seed):
    g = np.random.default_rng(seed)
    P = pos0 + T
    f = lambda *s: g.standard_normal(s).astype(np.float32)
    return f(T, H, dn), f(P, G, dn), f(P, G, dv)


@pytest.mark.parametrize("T,pos0,H,G,dn,dv", [(64, 0, 2, 2, 64, 64), (65, 31, 4, 1, 60, 36), (33, 200, 8, 4, 128, 128), (97, 3, 3, 3, 72, 128), (40, 0, 16, 8, 192, 100), (70, 0, 1, 1, 130, 20),
                                              (66, 5, 2, 1, 33, 17), (128, 64, 8, 8, 16, 16), (200, 0, 5, 5, 40, 64), (256, 0, 16, 4, 128, 128)])
@pytest.mark.parametrize("option", ["plain", "window", "chunks", "keep", "cap_sink", "slopes"])
def test_window_attention_of_a_portion(T, pos0, H, G, dn, dv, option):
    q, k, v = values(T, pos0, H, G, dn, dv, T + dn)
    kw, ref = {}, {}
    if option == "window":
        kw, ref = {"window": 37}, {"window": 37}
    elif option == "chunks":
        kw, ref = {"window": 48, "chunks": True}, {"window": 48, "chunks": True}
    elif option == "keep":
        kw, ref = {"window": 20, "keep_first": 5}, {"window": 20, "keep": 5}
    elif option == "cap_sink":
        kw, ref = {"softcap": 3.0, "sink": True}, {"cap": 3.0, "sinks": np.zeros(H)}
    elif option == "slopes":
        sl = np.exp2(-8.0 * (np.arange(H) + 1) / H).astype(np.float32)
        kw, ref = {"slopes": sl}, {"slopes": sl.astype(np.float64)}
    cache = np.concatenate([k.reshape(k.shape[0], -1), v.reshape(v.shape[0], -1)], 1)
    got = Lr.window_attention(q.reshape(T, -1), cache, H, G, 1, dn, dv, pos0, kw.pop("window", 0), 1.0 / np.sqrt(dn), split=False, **kw)
    want = reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), pos0, 1.0 / np.sqrt(dn), **ref)
    assert np.abs(got.reshape(T, H, dv) - want).max() < 2e-5 * np.abs(v).max()


def test_a_towering_key_and_huge_scores():
    T, H, dn, dv = 100, 2, 64, 64
    q, k, v = values(T, 0, H, H, dn, dv, 1)
    k[41] *= 60.0                              # scores of several hundred: every other weight vanishes
    cache = np.concatenate([k.reshape(T, -1), v.reshape(T, -1)], 1)
    got = Lr.window_attention(q.reshape(T, -1), cache, H, H, 1, dn, dv, 0, 0, 1.0, split=False)
    want = reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), 0, 1.0)
    err = np.abs(got.reshape(T, H, dv) - want)
    assert np.isfinite(got).all() and err.max() < 2e-3      # (scores up to ~500: 2^-24 * 68 * sum |q k| = 5e-3 of a weight between near-ties)


@pytest.mark.parametrize("R,dr,H", [(12, 0, 1), (16, 4, 3), (500, 30, 16), (512, 64, 16), (64, 8, 17)])
@pytest.mark.parametrize("T,pos0,window", [(1, 0, 0), (1, 63, 0), (1, 1300, 0), (1, 700, 129), (2, 64, 1), (7, 300, 64)])
def test_decoded_tokens_over_shared_latents_at_the_edges(R, dr, H, T, pos0, window):
    """the form whose keys are the latents themselves: ranks off the operand sizes, no rotated part, one head and more heads than a tile, one key, windows, many splits"""
    g = np.random.default_rng(R + T + pos0)
    n = pos0 + T
    q, cache = g.standard_normal((T, H, R + dr)).astype(np.float32), g.standard_normal((n, R + dr)).astype(np.float32)
    scale = (R + dr) ** -0.5
    got = Lr.latent_attention(q.reshape(T, -1), cache, R, dr, H, pos0, window, scale).reshape(T, H, R)
    for t in range(T):
        lo = max(0, pos0 + t - window + 1) if window else 0
        keys = cache[lo:pos0 + t + 1].astype(np.float64)
        s = q[t].astype(np.float64) @ keys.T * scale
        p = np.exp(s - s.max(axis=1, keepdims=True))
        want = (p / p.sum(axis=1, keepdims=True)) @ keys[:, :R]
        assert np.abs(got[t] - want).max() < 2e-5 * np.abs(keys).max()


@pytest.mark.parametrize("R,dr", [(128, 0), (120, 8), (129, 0), (125, 4), (320, 0), (256, 64), (321, 0), (300, 21)])
@pytest.mark.parametrize("T,H,pos0,window", [(1, 1, 0, 0), (3, 5, 95, 0), (8, 16, 200, 70)])
def test_shared_latents_at_the_limits_of_the_operand_sizes(R, dr, H, T, pos0, window):
    """keys of 128 and 320 entries and one past them, with and without a rotated part"""
    test_decoded_tokens_over_shared_latents_at_the_edges(R, dr, H, T, pos0, window)
