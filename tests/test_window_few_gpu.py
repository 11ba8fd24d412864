"""Window attention of a few decoded tokens (csrc/window_attention.hip, window_attention_few_kernel) against float64: chunks of 64 keys at their edges, one workgroup and several parts,
every option of the scores and the result, heads per key / value head from one to eight.  Bound as for the prompts' form: 2e-5 of the largest value."""
import numpy as np
import pytest

from ntransformer_amd import layers as Lr
from test_attention_tile_gpu import reference, values

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,pos0,H,G,dn,dv", [(1, 0, 1, 1, 4, 4), (1, 63, 4, 1, 128, 128), (2, 63, 6, 3, 64, 36), (8, 100, 16, 4, 128, 128), (1, 255, 8, 1, 100, 128), (1, 256, 16, 8, 128, 60),
                                              (3, 700, 5, 5, 68, 128), (1, 4500, 14, 2, 128, 128), (8, 1500, 32, 8, 128, 128)])
@pytest.mark.parametrize("option", ["plain", "window", "chunks", "keep", "cap_sink", "slopes", "rel", "gate", "norm"])
def test_few_tokens(T, pos0, H, G, dn, dv, option):
    q, k, v = values(T, pos0, H, G, dn, dv, T + dn)
    g = np.random.default_rng(7)
    kw, ref, factor = {}, {}, 1.0
    if option == "window":
        kw, ref = {"window": 70}, {"window": 70}
    elif option == "chunks":
        kw, ref = {"window": 96, "chunks": True}, {"window": 96, "chunks": True}
    elif option == "keep":
        kw, ref = {"window": 40, "keep_first": 30}, {"window": 40, "keep": 30}
    elif option == "cap_sink":
        sk = g.standard_normal(H).astype(np.float32)
        kw, ref = {"softcap": 3.0, "sinks": sk}, {"cap": 3.0, "sinks": sk.astype(np.float64)}
    elif option == "slopes":
        sl = np.exp2(-8.0 * (np.arange(H) + 1) / H).astype(np.float32)
        kw, ref = {"slopes": sl}, {"slopes": sl.astype(np.float64)}
    elif option == "rel":
        kw = {"rel": g.standard_normal((5, H)).astype(np.float32), "bucket_of": np.minimum(np.arange(40) // 3, 4).astype(np.int32)}
        ref = {"rel": kw["rel"].astype(np.float64), "bucket_of": kw["bucket_of"]}
    elif option == "gate":
        kw = {"gate": g.standard_normal((T, H * dv)).astype(np.float32)}
        factor = (1.0 / (1.0 + np.exp(-kw["gate"].astype(np.float64)))).reshape(T, H, dv)
    elif option == "norm":
        kw = {"sub_norm": True, "out_scale": 0.7}
    cache = np.concatenate([k.reshape(k.shape[0], -1), v.reshape(v.shape[0], -1)], 1)
    want = reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), pos0, 1.0 / np.sqrt(dn), **ref) * factor
    if option == "norm":
        want = want / np.sqrt((want ** 2).mean(2, keepdims=True) + 1e-6) * 0.7
    window = kw.pop("window", 0)
    for split in (True, False):
        got = Lr.window_attention(q.reshape(T, -1), cache, H, G, 1, dn, dv, pos0, window, 1.0 / np.sqrt(dn), split=split, **kw).reshape(T, H, dv)
        assert np.abs(got - want).max() < 2e-5 * max(np.abs(v).max(), np.abs(want).max()), split


# two chunks and the first keys of a third, with more and fewer heads a key; eight tokens of eight heads a key on either side of 256 and 2048 keys
@pytest.mark.parametrize("T,pos0,H,G,dn,dv", [(1, 64, 8, 1, 128, 128), (1, 127, 4, 1, 128, 64), (3, 125, 6, 2, 64, 64), (1, 127, 4, 2, 64, 64), (1, 128, 4, 4, 64, 64), (2, 128, 4, 2, 64, 64),
                                              (8, 248, 64, 8, 64, 64), (8, 249, 64, 8, 64, 64), (7, 300, 56, 8, 64, 64), (8, 2040, 32, 4, 64, 64), (8, 2041, 32, 4, 64, 64)])
def test_where_the_keys_are_cut(T, pos0, H, G, dn, dv):
    test_few_tokens(T, pos0, H, G, dn, dv, "cap_sink")


@pytest.mark.parametrize("what", [np.nan, np.inf])
def test_only_visible_positions_matter(what):
    T, pos0, H, G, dn, dv = 2, 90, 4, 2, 64, 64
    q, k, v = values(T, pos0, H, G, dn, dv, 3)
    v[5], k[7], v[91, 0, 3] = what, what, what              # the first two lie ahead of the window, the last is the second token's own
    cache = np.concatenate([k.reshape(k.shape[0], -1), v.reshape(v.shape[0], -1)], 1)
    got = Lr.window_attention(q.reshape(T, -1), cache, H, G, 1, dn, dv, pos0, 50, 0.125).reshape(T, H, dv)
    bad = np.zeros(got.shape, bool)
    bad[1, :2, 3] = True
    assert np.array_equal(~np.isfinite(got), bad)


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("pos0", [20, 48, 400, 1500])
@pytest.mark.parametrize("kind", ["query", "every key", "last key", "key alone in its sixteen", "value without weight"])
@pytest.mark.parametrize("sink", [None, -1.0])
def test_what_is_not_a_number_stays_one(kind, pos0, split, sink):
    """a query or a visible key of NaN makes a head's results NaN (no row of zeros), as an infinite value does whose weight has underflowed (0 * inf)"""
    H, G, dn, dv = 4, 2, 64, 64
    q, k, v = values(1, pos0, H, G, dn, dv, 3)
    bad = np.zeros((1, H, dv), bool)
    bad[0, :2] = True
    if kind == "query":
        q[0, 1, 5] = np.nan
        bad[0, 0] = False
    elif kind == "every key":
        k[:, 0, 5] = np.nan
    elif kind == "last key":
        k[pos0, 0, 5] = np.nan
    elif kind == "key alone in its sixteen":
        pos0 = pos0 // 16 * 16                  # the token's own key begins a group of sixteen
        k, v = k[:pos0 + 1], v[:pos0 + 1]
        k[pos0, 0, 5] = np.nan
    else:
        q[:, :, 0], k[3, 0], k[3, 0, 0] = 1.0, 0.0, -8000.0
        v[3, 0, 7] = np.inf
        bad[:] = False
        bad[0, :2, 7] = True
    cache = np.concatenate([k.reshape(k.shape[0], -1), v.reshape(v.shape[0], -1)], 1)
    kw = {"sinks": np.full(H, sink, np.float32)} if sink is not None else {}
    got = Lr.window_attention(q.reshape(1, -1), cache, H, G, 1, dn, dv, pos0, 0, 0.125, split=split, **kw).reshape(1, H, dv)
    assert np.array_equal(np.isnan(got), bad)
    assert np.isfinite(got[~bad]).all()
