"""GGUF prompts through the routes that a pass chooses by the model's sizes, the number of tokens and the position of the first.  Against the per-token sequence (every matrix a token at a time, every
layer whole), the prompt's logits and those of tokens decoded behind it, which read every cache row.  Caches of halves: a value at a rounding boundary falls to either side, 1e-3 (2e-4 seen)."""
import numpy as np
import pytest

from ntransformer_amd import engine as E
from oracle import arbiter
from oracle import oracle as O

pytestmark = pytest.mark.gpu
REL = 1e-3


def rel(got, ref):
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    return float(np.sqrt(np.mean((got - ref) ** 2)) / (np.sqrt(np.mean(ref ** 2)) + 1e-30))


def spec(hidden, inter, heads, kv_heads, mix, layers=2, ctx=2048):
    return E.SynthSpec(hidden, inter, layers, heads, kv_heads, 512, ctx, 1e-5, 500000.0, 256, 257, mix.encode(), 3)


def passes(s, ctx, portions, batched, decode=2):
    """logits of the portions one behind the other, then of `decode` single tokens"""
    toks = [int(t) for t in np.random.default_rng(sum(portions)).integers(0, s.vocab, sum(portions) + decode)]
    e = E.Engine()
    e.load_synthetic(s, ctx)
    e.set_option("batched_prefill", batched)
    at, out = 0, []
    for n in portions:
        out.append(e.forward(toks[at:at + n], at))
        at += n
    out += [e.decode_fused(t, at + i, False) for i, t in enumerate(toks[at:])]
    e.close()
    return np.stack(out)


def check(s, ctx, portions, decode=2):
    got, want = passes(s, ctx, portions, 1, decode), passes(s, ctx, portions, 0, decode)
    assert np.isfinite(want).all() and np.isfinite(got).all() and rel(got, want) < REL


@pytest.mark.parametrize("mix", ["Q8_0", "Q4_K_M"])
@pytest.mark.parametrize("T", [2, 4, 16, 17, 33])
def test_heads_of_512(mix, T):
    """wider than the launch that rotates from the projections' sums"""
    check(spec(2048, 1024, 4, 2, mix), 128, [T])


@pytest.mark.parametrize("mix,T", [("Q8_0", 40), ("Q6_K", 17), ("F16", 40)])
def test_contexts_beyond_the_decoding_attention(mix, T):
    """heads of 96 entries in a context of 65536: the launch of a decoded token keeps scores for all of it, a prompt's for the keys that are there"""
    check(spec(768, 1024, 8, 2, mix, ctx=65536), 65536, [T], decode=0)


def test_rows_beyond_the_decoding_products(tmp_path):
    """33024 inputs, more than the product of a single token takes: against the oracle"""
    s, path = spec(256, 33024, 2, 1, "Q8_0"), str(tmp_path / "m.gguf")
    E.synth_write_gguf(path, s)
    toks = [int(t) for t in np.random.default_rng(1).integers(0, s.vocab, 40)]
    e = E.Engine()
    e.load(path, 64)
    got = e.forward(toks, 0)
    e.close()
    assert np.isfinite(got).all() and rel(got, O.OracleModel(path, 64).forward(toks, 0)) < REL


@pytest.mark.parametrize("T", [17, 40, 90])
def test_the_last_tokens_products_are_a_prompts(tmp_path, T):
    """the last layer's results for the last token are no further from 64 bits than those of a prompt whose layers are all whole (16 tokens): against the float64 arbiter over the engine's own cache
    rows, so that no rounding of a cached value counts.  1.5 times the error over three models (2.0 times and more where the inputs are rounded to 22 bits of their block's largest, 1.05 seen)"""
    def error(n):
        sq = []
        for seed in (1, 2, 3):
            s, path = spec(1024, 2048, 8, 2, "Q6_K", layers=1), str(tmp_path / ("%d.gguf" % seed))
            s.seed = seed
            E.synth_write_gguf(path, s)
            om = O.OracleModel(path, 128)
            per = om.nkv * om.hd
            toks = [int(t) for t in np.random.default_rng(seed * 100 + n).integers(0, s.vocab, n)]
            e = E.Engine()
            e.load(path, 128)
            got = e.forward(toks, 0).astype(np.float64)
            k, v = e.kv_read(0, 0, n, per)
            e.close()
            K, V = np.zeros_like(om.k_cache), np.zeros_like(om.v_cache)
            K[0][:n * per], V[0][:n * per] = k.reshape(-1), v.reshape(-1)
            sq.append(rel(got, arbiter.ArbiterModel(om).forward(toks, 0, (K, V))) ** 2)
        return np.sqrt(np.mean(sq))
    assert error(T) < 1.5 * error(16)


@pytest.mark.parametrize("mix", ["Q8_0", "Q4_K_M"])
@pytest.mark.parametrize("start", [5, 600])
@pytest.mark.parametrize("T", [2, 3, 4, 16, 17, 32, 33, 70])
def test_prompts_behind_a_context(mix, start, T):
    """a prompt that begins behind others: the short form's own rotation and attention (2 and 3 tokens: of whole projections), several formats' sums side by side, the last layer cut short; few and more
    positions in front than the single-pass attention of a decoded token walks"""
    check(spec(1024, 2048, 8, 2, mix), 1024, [start, T])


@pytest.mark.parametrize("T", [2, 5, 33, 70, 200])
@pytest.mark.parametrize("start", [0, 7])
def test_half_precision_chain(T, start):
    """from 3072 inputs on: the norm's halves from the launch that sums the projection in front of it, query, key and value rotated from their joined pieces, the last layer cut short from 33 tokens on"""
    check(spec(3072, 3200, 24, 8, "F16"), 256, [start, T] if start else [T])
