"""A prompt whose last token alone is wanted, or none: the last layer computes what later tokens attend to for all of its tokens and its result for the wanted one.  Every mixer that can come
last in the two families that do so, against the oracle and against the same prompt with every place wanted: the logits, and those of tokens decoded behind it (which read everything that the
last layer left behind).  9 to 11 tokens lie on both sides of the line from which on it is done; 70 tokens take the tiled products; portions with nothing wanted come first."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import fabolorn_oracle as FO  # noqa: E402
import fifotar_oracle as O  # noqa: E402
from ntransformer_amd.engine import Engine  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = {"float32": 2e-4, "bfloat16": 4e-2}     # (the families' own)


def rel(got, ref):
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    return float(np.sqrt(np.mean((got - ref) ** 2)) / (np.sqrt(np.mean(ref ** 2)) + 1e-30))


def check(oracle, cfg, tmp_path, dtype, T):
    w = oracle.random_weights(cfg, 5)
    folder = str(tmp_path / "m")
    oracle.save_model(folder, cfg, w)
    toks = [int(t) for t in np.random.default_rng(T).integers(0, cfg["vocab"], T + 3)]
    ref = oracle.forward(cfg, w, toks)
    ref = (ref[0] if isinstance(ref, tuple) else ref)
    ref = np.asarray(ref.numpy() if hasattr(ref, "numpy") else ref)
    e = Engine()
    e.load_folder(folder, max_context=T + 8, dtype=dtype, slots=1)

    def decoded(s):
        out = np.concatenate([e.seq_forward(s, [t], want=[0]) for t in toks[T:]])
        e.seq_release(s)
        return out
    s = e.seq_acquire()
    full = e.seq_forward(s, toks[:T])
    full = np.concatenate([full[-1:], decoded(s)])
    s = e.seq_acquire()
    last = e.seq_forward(s, toks[:T], want=[T - 1])
    last = np.concatenate([last, decoded(s)])
    s = e.seq_acquire()
    e.seq_forward(s, toks[:T], want=[])
    none = decoded(s)
    assert rel(last, ref[T - 1:]) < TOL[dtype] and rel(none, ref[T:]) < TOL[dtype]
    same = 1e-5 if dtype == "float32" else TOL[dtype]      # (32 bits: other orders of the same sums)
    assert rel(last, full) < same and rel(none, full[1:]) < same
    if T > 20:                                             # in portions, the first with nothing wanted
        s = e.seq_acquire()
        e.seq_forward(s, toks[:13], want=[])
        last = np.concatenate([e.seq_forward(s, toks[13:T], want=[T - 14]), decoded(s)])
        assert rel(last, ref[T - 1:]) < TOL[dtype] and rel(last, full) < same
    e.close()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T", [9, 10, 11, 70])
@pytest.mark.parametrize("last", ["attention", "delta", "latent", "alone"])
def test_scaled_form(tmp_path, dtype, T, last):
    layers = {"attention": [O.attention_layer(size=24), O.delta_layer(), O.attention_layer(size=24, ff=64)], "delta": [O.attention_layer(size=24), O.delta_layer(ff=20)],
              "latent": [O.delta_layer(), O.latent_layer(kv_rank=64)], "alone": [O.attention_layer(size=24)]}[last]
    check(O, O.config(layers, width=64), tmp_path, dtype, T)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T", [9, 10, 11, 70])
@pytest.mark.parametrize("kw", [dict(), dict(layers=("latent_attention_2",)), dict(layers=("latent_attention", "latent_attention_2"), loop=(0, 2, 2)), dict(mlp_on=(True, False))])
def test_parallel_form(tmp_path, dtype, T, kw):
    check(FO, FO.small_config(**kw), tmp_path, dtype, T)


@pytest.mark.parametrize("last", ["20480", "40960", "latent"])
def test_last_layers_beyond_a_decoded_tokens_launches(tmp_path, last):
    """a unit of 40960 values, keys of 820 entries: what the products and the attention of a few tokens refuse, a prompt's take, its last layer whole (of 20480 values they take)"""
    layers = {"20480": [O.attention_layer(size=24), O.attention_layer(size=24, ff=20480)], "40960": [O.attention_layer(size=24), O.attention_layer(size=24, ff=40960)], "latent": [O.latent_layer(heads=2, dim=8, rot_dim=308, kv_rank=512)]}[last]
    cfg = O.config(layers, width=64)
    w = O.random_weights(cfg, 5)
    O.save_model(str(tmp_path / "m"), cfg, w)
    toks = [int(t) for t in np.random.default_rng(3).integers(0, cfg["vocab"], 16)]
    e = Engine()
    e.load_folder(str(tmp_path / "m"), max_context=32, dtype="float32", slots=1)
    got = e.seq_forward(e.seq_acquire(), toks, want=[15])
    e.close()
    assert rel(got, O.forward(cfg, w, toks)[0][15:]) < TOL["float32"]


@pytest.mark.parametrize("mix", ["Q8_0", "Q4_K_M", "F16"])
@pytest.mark.parametrize("T", [32, 33, 70])
def test_gguf_prompts(mix, T):
    """against the per-token sequence, which runs every layer for every token: the prompt's logits, and those of tokens decoded behind it (which read the last layer's cache rows).  Caches of
    halves: a value at a rounding boundary falls to either side, 1e-3 (2e-4 seen)"""
    from ntransformer_amd import engine as E
    spec = E.synth_spec("small", mix, seed=3, layers=2)
    toks = [int(t) for t in np.random.default_rng(T).integers(0, 2048, T + 3)]
    out = []
    for batched in (1, 0):
        e = E.Engine()
        e.load_synthetic(spec, 128)
        e.set_option("batched_prefill", batched)
        lg = [e.forward(toks[:T], 0)]
        lg += [e.decode_fused(t, T + i, False) for i, t in enumerate(toks[T:])]
        e.close()
        out.append(np.stack(lg))
    assert np.isfinite(out[0]).all() and rel(out[0], out[1]) < 1e-3


@pytest.mark.parametrize("mix", ["Q6_K", "Q4_K_M", "Q8_0"])
@pytest.mark.parametrize("T", [16, 17])
def test_gguf_prompts_beside_the_short_form(mix, T):
    """(formats that layers_short takes up to 16 tokens only; 1e-3 as above)"""
    test_gguf_prompts(mix, T)
