"""GGUF prompts through the routes that a pass chooses by the model's sizes, the number of tokens and the position of the first.  Against the per-token sequence (every matrix a token at a time, every
layer whole), the prompt's logits and those of tokens decoded behind it, which read every cache row.  Caches of halves: a value at a rounding boundary falls to either side, 1e-3 (2e-4 seen)."""
import numpy as np
import pytest

from ntransformer_amd import engine as E

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
