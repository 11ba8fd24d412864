"""The prompt attention on bfloat16 matrix instructions (csrc/attention_pieces.hip.h): everything that is asked of the 32-bit form, with room for the pieces, then the edges of its own tiles
(64 rows, pairs of 32 positions, positions that stay visible ahead of a window) and its error beside the 32-bit form's."""
import functools

import numpy as np
import pytest

from ntransformer_amd import layers as Lr
from test_attention_tile_gpu import (reference, values, test_latent_values_that_are_not_finite_stay_with_the_rows_that_see_them,  # noqa: F401
                                     test_values_that_are_not_finite_stay_with_the_rows_that_see_them, test_window_attention_of_a_portion)

pytestmark = pytest.mark.gpu
window_f32, latent_f32 = Lr.window_attention, Lr.latent_attention


@pytest.fixture(autouse=True)
def _halves(monkeypatch):
    monkeypatch.setattr(Lr, "window_attention", functools.partial(window_f32, halves=True))
    monkeypatch.setattr(Lr, "latent_attention", functools.partial(latent_f32, halves=True))


def attend(form, q, k, v, G, pos0, **kw):
    T, H, dn = q.shape
    cache = np.concatenate([k.reshape(k.shape[0], -1), v.reshape(v.shape[0], -1)], 1)
    return form(q.reshape(T, -1), cache, H, G, 1, dn, v.shape[2], pos0, kw.pop("window", 0), kw.pop("scale", dn ** -0.5), split=False, **kw).reshape(T, H, v.shape[2])


# rows off 64, positions off 32 and off pairs of tiles, one pair and an odd number of tiles, a window that starts inside a tile, kept positions that reach into it
@pytest.mark.parametrize("T,pos0,H,G,dn,dv", [(64, 0, 1, 1, 65, 1), (32, 0, 4, 2, 192, 128), (33, 95, 2, 1, 100, 128), (65, 64, 8, 8, 128, 127), (130, 1, 3, 1, 72, 33), (96, 160, 16, 16, 191, 64)])
@pytest.mark.parametrize("window,keep,chunks", [(0, 0, False), (1, 0, False), (33, 0, False), (70, 40, False), (20, 100, False), (64, 0, True), (45, 0, True)])
def test_edges_of_rows_tiles_and_windows(T, pos0, H, G, dn, dv, window, keep, chunks):
    q, k, v = values(T, pos0, H, G, dn, dv, T + dn)
    got = attend(Lr.window_attention, q, k, v, G, pos0, window=window, keep_first=keep, chunks=chunks)
    want = reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), pos0, dn ** -0.5, window, chunks, keep)
    assert np.abs(got - want).max() < 2e-5 * np.abs(v).max()


@pytest.mark.parametrize("dn", [72, 128, 192])
@pytest.mark.parametrize("kind", ["normal", "towering", "wide"])
def test_no_further_from_float64_than_the_32_bit_form(dn, kind):
    """root mean square over 200 x 4 x 128 results, so known to a fraction of a percent"""
    T, H, pos0 = 200, 4, 300
    q, k, v = values(T, pos0, H, H, dn, 128, dn)
    if kind == "towering":                     # a few channels tower over the others, a few positions over theirs
        q[:, :, ::37] *= 20.0
        k[:, :, ::23] *= 15.0
        v[::29] *= 300.0
    elif kind == "wide":
        k *= np.exp2(np.random.default_rng(1).integers(-3, 4, (pos0 + T, 1, 1))).astype(np.float32)
        v *= np.exp2(np.random.default_rng(2).integers(-12, 12, (pos0 + T, 1, 1))).astype(np.float32)
    scale = dn ** -0.5 * (0.05 if kind == "towering" else 1.0)
    want = reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), pos0, scale)
    err = [np.linalg.norm(attend(f, q, k, v, H, pos0, scale=scale) - want) for f in (Lr.window_attention, window_f32)]
    print(dn, kind, "error as pieces %.3g, in 32 bits %.3g" % tuple(e / np.linalg.norm(want) for e in err))
    assert err[0] <= 1.03 * err[1]


@pytest.mark.parametrize("T,pos0,window", [(32, 0, 0), (100, 41, 0), (70, 50, 42), (64, 300, 129)])
def test_two_part_keys_behind_a_first_position(T, pos0, window):
    H, R, dr, dn, dv = 3, 24, 16, 112, 80
    g = np.random.default_rng(T)
    f = lambda *s: g.standard_normal(s).astype(np.float32)
    key0 = max(0, pos0 - window + 1) if window else 0
    q, cache, k, v = f(T, H, dn + dr), f(pos0 + T, R + dr), f(pos0 + T - key0, H, dn), f(pos0 + T - key0, H, dv)
    got = Lr.latent_attention(q.reshape(T, -1), cache, R, dr, H, pos0, window, (dn + dr) ** -0.5, K=k.reshape(len(k), -1), V=v.reshape(len(v), -1), key0=key0).reshape(T, H, dv)
    keys = np.concatenate([np.zeros((key0, H, dn + dr)), np.concatenate([k, np.repeat(cache[key0:, None, R:], H, 1)], 2)]).astype(np.float64)
    want = reference(q.astype(np.float64), keys, np.concatenate([np.zeros((key0, H, dv)), v]).astype(np.float64), pos0, (dn + dr) ** -0.5, window)
    assert np.abs(got - want).max() < 2e-5 * np.abs(v).max()


def test_values_of_every_magnitude_and_rows_of_zeros():
    T, H = 90, 2
    for power in (-120, -30, 30, 100):
        q, k, v = values(T, 0, H, H, 96, 40, 1)
        v = np.ldexp(v, power).astype(np.float32)
        k[3], q[5], v[7], v[32:64] = 0.0, 0.0, 0.0, 0.0
        got = attend(Lr.window_attention, q, k, v, H, 0)
        want = reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), 0, 96 ** -0.5)
        assert np.abs(got - want).max() < 2e-5 * np.abs(v).max() + 1e-37
        k2, q2 = np.ldexp(k, power).astype(np.float32), np.ldexp(q, -power).astype(np.float32)       # the same scores
        assert np.abs(attend(Lr.window_attention, q2, k2, v, H, 0) - want).max() < 2e-5 * np.abs(v).max() + 1e-37


@pytest.mark.parametrize("what", [np.nan, np.inf, -np.inf])
def test_keys_that_are_not_finite(what):
    """a key's -inf (or +inf against a negative query) is a weight of zero, a NaN or a score of +inf makes the rows that see it NaN, and no other row"""
    T, H, dn = 80, 2, 128
    q, k, v = values(T, 0, H, H, dn, 64, 5)
    k[40, 0, 3] = what
    got, want = attend(Lr.window_attention, q, k, v, H, 0), attend(window_f32, q, k, v, H, 0)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.nanmax(np.abs(got - want)) < 2e-5 * np.abs(v).max()


# ... and with two heads a key: from 64 rows on such portions take this form whatever they see
@pytest.mark.parametrize("T,pos0,H,G,dn,dv", [(32, 0, 2, 1, 65, 1), (33, 95, 4, 2, 100, 128), (130, 1, 6, 3, 72, 33), (96, 160, 32, 16, 191, 64), (9, 40, 8, 1, 128, 100)])
@pytest.mark.parametrize("window,keep,chunks", [(0, 0, False), (1, 0, False), (33, 0, False), (70, 40, False), (20, 100, False), (64, 0, True), (45, 0, True)])
def test_edges_with_heads_that_share_keys(T, pos0, H, G, dn, dv, window, keep, chunks):
    test_edges_of_rows_tiles_and_windows(T, pos0, H, G, dn, dv, window, keep, chunks)


@pytest.mark.parametrize("power", [20, 40, 100])
@pytest.mark.parametrize("kind", ["later", "left of the window", "earlier, without weight", "leading rows", "value columns", "query and key channels"])
@pytest.mark.parametrize("dn", [128, 192])
def test_every_row_at_the_error_of_what_it_sees(kind, power, dn):
    """Sizes that differ by 2^power within a tile: between positions, seen by a row or not, between columns of the values, between channels of queries and keys.  Every row's error over sum(weight |value|)
    of that row, column by column: the largest is no more than 1.5 of the 32-bit form's largest (two of 30000 numbers of the same distribution)."""
    T, H, pos0, window = 120, 2, 70, 0
    q, k, v = values(T, pos0, H, 1, dn, 128, power + dn)
    big = np.float32(2.0 ** power)
    if kind == "later":
        v[pos0 + 40] *= big                     # positions pos0 + 32 .. 39 share its tile, those behind it see it
        v[pos0 + T - 1] *= big
    elif kind == "left of the window":
        window = 50
        v[[24, 61, 90, 125]] *= big
    elif kind == "earlier, without weight":     # seen by all, scores of about -150 and lower
        k[[3, 80]], q[:, :, 0] = 0.0, 1.0
        k[[3, 80], :, 0] = -150.0 * dn ** 0.5
        v[[3, 80]] *= big
    elif kind == "leading rows":
        v[:100] /= big
    elif kind == "value columns":
        v[:, :, ::3] *= big
    else:
        s = np.exp2(np.random.default_rng(power).integers(-(power // 2), power // 2, dn)).astype(np.float32)
        q, k = (q * s).astype(np.float32), (k / s).astype(np.float32)
    f64 = lambda a: a.astype(np.float64)
    want, size = (reference(f64(q), f64(k), f64(x), pos0, dn ** -0.5, window) for x in (v, np.abs(v)))
    err = [(np.abs(attend(f, q, k, v, 1, pos0, window=window) - want) / size).max() for f in (Lr.window_attention, window_f32)]
    print(kind, power, dn, "as pieces %.3g, in 32 bits %.3g" % tuple(err))
    assert err[0] <= 1.5 * err[1]


@pytest.mark.parametrize("low", [-np.inf, np.finfo(np.float32).min, -3e38])
def test_scores_of_the_types_lowest_value(low):
    """a bias of the lowest value on the nearest distances: rows that see nothing else weigh all of it alike (-inf: not at all), the others give it no weight"""
    T, H, dn = 100, 2, 96
    q, k, v = values(T, 0, H, 1, dn, 64, 8)
    rel, bucket_of = np.array([[low] * H, [0.25] * H], np.float32), (np.arange(60) > 40).astype(np.int32)
    got = attend(Lr.window_attention, q, k, v, 1, 0, rel=rel, bucket_of=bucket_of)
    assert np.abs(got - attend(window_f32, q, k, v, 1, 0, rel=rel, bucket_of=bucket_of)).max() < 2e-5 * np.abs(v).max()
    mean = np.cumsum(v.astype(np.float64), 0) / np.arange(1, T + 1)[:, None, None]
    assert np.abs(got[:41] - (0.0 if low == -np.inf else mean[:41])).max() < 2e-5 * np.abs(v).max()
