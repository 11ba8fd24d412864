"""The matrix-instruction form of the prompt attention (csrc/attention_tile.hip.h) at the edges of its tiles (32 rows, 32 keys, head sizes below, at and between its operand
sizes) against float64: every option of the window mixer that it takes, and the latent mixer's two-part keys.  Bound on a result: scores are off by (dk + 4) * 2^-24 of
sum |q k| (at most ~30 here), weights by that and an exponential's rounding, the weighted sum by its (keys + 4) additions: 2e-5 of the largest value."""
import numpy as np
import pytest

from ntransformer_amd import layers as Lr

pytestmark = pytest.mark.gpu


def reference(q, k, v, pos0, scale, window=0, chunks=False, keep=0, cap=0.0, sinks=None, slopes=None, rel=None, bucket_of=None):
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
            if rel is not None:
                s = s + rel[bucket_of[np.clip(p - j, 0, len(bucket_of) - 1)], h]
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


@pytest.mark.parametrize("R,dr", [(256, 60), (260, 60), (252, 68), (512, 128), (509, 131), (512, 132), (512, 304), (64, 752)])
@pytest.mark.parametrize("T,H,pos0,window", [(1, 17, 31, 0), (4, 8, 32, 0), (2, 16, 4500, 0)])
def test_shared_latents_by_rank_and_by_key(R, dr, H, T, pos0, window):
    """four and eight waves (a rank of 256 and one past it, keys of 320), keys of 640, the longest ones; the last position of a tile, the first of the next, several tiles a workgroup"""
    test_decoded_tokens_over_shared_latents_at_the_edges(R, dr, H, T, pos0, window)


@pytest.mark.parametrize("what", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("H,G,dn,dv,window,keep,option", [(2, 2, 64, 64, 0, 0, ""), (4, 1, 33, 17, 0, 0, "gate"), (2, 1, 128, 128, 20, 3, "cap_sink"), (3, 3, 192, 100, 33, 0, "slopes"),
                                                          (4, 2, 40, 64, 48, 0, "chunks"), (2, 1, 16, 33, 0, 0, "rel"), (3, 1, 128, 36, 37, 0, "head_gate")])
def test_values_that_are_not_finite_stay_with_the_rows_that_see_them(H, G, dn, dv, window, keep, option, what):
    """a position's value reaches the tokens it is visible to and no other, whatever shares their tiles, under every option of the scores and of the result; a visible one follows the
    arithmetic (inf - inf, 0 * inf)"""
    T, pos0 = 90, 7
    q, k, v = values(T, pos0, H, G, dn, dv, 3)
    g = np.random.default_rng(4)
    k[60] -= 40.0 * q[55].mean(0)              # (a weight that may vanish in 32 bits)
    for at, col in ((60, 1), (60, 9), (77, 16), (2, 4)):
        v[at, 0, col] = what
    v[61, 0, 9] = -what
    kw, ref, factor = {}, {}, np.ones((T, H, dv))
    if option == "cap_sink":
        sk = g.standard_normal(H).astype(np.float32)
        kw, ref = {"softcap": 3.0, "sinks": sk}, {"cap": 3.0, "sinks": sk.astype(np.float64)}
    elif option == "slopes":
        sl = np.exp2(-8.0 * (np.arange(H) + 1) / H).astype(np.float32)
        kw, ref = {"slopes": sl}, {"slopes": sl.astype(np.float64)}
    elif option == "rel":
        kw = {"rel": g.standard_normal((5, H)).astype(np.float32), "bucket_of": np.minimum(np.arange(40) // 3, 4).astype(np.int32)}
        ref = {"rel": kw["rel"].astype(np.float64), "bucket_of": kw["bucket_of"]}
    elif "gate" in option:
        gt = g.standard_normal((T, H if option == "head_gate" else H * dv)).astype(np.float32)
        kw = {"gate": gt, "head_gate": option == "head_gate"}
        factor = np.broadcast_to(1.0 / (1.0 + np.exp(-gt.astype(np.float64))).reshape(T, H, -1), (T, H, dv))
    chunks = option == "chunks"
    cache = np.concatenate([k.reshape(k.shape[0], -1), v.reshape(v.shape[0], -1)], 1)
    got = Lr.window_attention(q.reshape(T, -1), cache, H, G, 1, dn, dv, pos0, window, 1.0 / np.sqrt(dn), split=False, keep_first=keep, chunks=chunks, **kw).reshape(T, H, dv)
    clean = np.where(np.isfinite(v), v, 0.0).astype(np.float64)
    want = reference(q.astype(np.float64), k.astype(np.float64), clean, pos0, 1.0 / np.sqrt(dn), window, chunks, keep, **ref) * factor
    j = np.arange(pos0 + T)
    for t in range(T):
        p = pos0 + t
        seen = (j <= p) & (((j // window == p // window) if chunks else (p - j < window)) | (j < keep) if window else True)
        for h in range(H):
            bad = (~np.isfinite(v[:, h // (H // G)]) & seen[:, None]).any(axis=0)
            assert np.abs(got[t, h, ~bad] - want[t, h, ~bad]).max() < 2e-5 * np.abs(clean).max(), (t, h)
            assert not np.isfinite(got[t, h, bad]).any(), (t, h)


@pytest.mark.parametrize("what", [np.nan, np.inf])
def test_latent_values_that_are_not_finite_stay_with_the_rows_that_see_them(what):
    """the two-part keys of the expanded latent form, behind a first position that is not zero"""
    T, pos0, key0, H, R, dr, dn, dv = 70, 50, 9, 2, 24, 8, 40, 48
    g = np.random.default_rng(5)
    f = lambda *s: g.standard_normal(s).astype(np.float32)
    q, cache, k, v = f(T, H, dn + dr), f(pos0 + T, R + dr), f(pos0 + T - key0, H, dn), f(pos0 + T - key0, H, dv)
    v[77 - key0, 1, 20] = what
    got = Lr.latent_attention(q.reshape(T, -1), cache, R, dr, H, pos0, 42, (dn + dr) ** -0.5, K=k.reshape(len(k), -1), V=v.reshape(len(v), -1), key0=key0).reshape(T, H, dv)
    keys = np.concatenate([np.zeros((key0, H, dn + dr)), np.concatenate([k, np.repeat(cache[key0:, None, R:], H, 1)], 2)]).astype(np.float64)
    clean = np.concatenate([np.zeros((key0, H, dv)), np.where(np.isfinite(v), v, 0.0)]).astype(np.float64)
    want = reference(q.astype(np.float64), keys, clean, pos0, (dn + dr) ** -0.5, 42)
    hit = np.zeros(got.shape, bool)
    hit[77 - pos0:77 - pos0 + 42, 1, 20] = True
    assert np.abs(got[~hit] - want[~hit]).max() < 2e-5 * np.abs(clean).max() and not np.isfinite(got[hit]).any()


@pytest.mark.parametrize("R,dr", [(1, 0), (2, 2), (3, 0), (3, 126), (2, 400), (9, 0), (31, 6), (125, 3), (127, 2), (255, 30), (510, 30), (511, 300)])
@pytest.mark.parametrize("T,H,pos0,window", [(1, 3, 0, 0), (2, 8, 33, 0), (3, 5, 700, 90)])
def test_shared_latents_of_rows_off_four_entries(R, dr, H, T, pos0, window):
    """rows that are no whole fours: entry by entry (up to 128) and in fours with the last ones moved, ranks below four beside rotated entries"""
    test_decoded_tokens_over_shared_latents_at_the_edges(R, dr, H, T, pos0, window)
